// lsgpu_trace.h -- closest-hit BVH4 traversal for one ray per lane (gfx950).
//
// Near-child-first stack traversal over 128-byte BVH4 nodes whose child boxes are
// inflated by a DELTA_BSP-sized margin, so node culling is conservative and the
// result depends only on the per-triangle SRLNP test (IntersectBspFast.cpp:189-252)
// and the plane distance (:349-352): among accepted triangles with distance in
// [box-clipped rayLengthMin, current best], the smallest distance wins, ties to the
// lowest triangle index -- independent of traversal order.
//
// A Filter plays the role of RRCollisionHandler::collides (RRCollider.h:59): it
// sees each candidate (triangle, side, distance, hitPoint2d) and may reject it, and it
// may end the search early or narrow the interval once a hit is accepted.
#pragma once
#include "lsgpu_internal.h"

namespace lsg {

struct TraceResult { int tri; float t, u, v; bool front; uint32_t slot; };

struct NoFilter {
    __device__ bool accept(uint32_t, bool, float, float, float) const { return true; }
    // after accepting a hit at t: true = stop searching
    __device__ bool done(float) const { return false; }
    // after accepting a hit: upper bound of the interval still worth searching
    __device__ float clamp(float best) const { return best; }
};

constexpr int32_t kDone = 0x7fffffff;          // never a node index: the ray is finished
constexpr uint32_t kNoSlot = 0xffffffffu;

// One lane's traversal stack: a column of a workgroup's LDS array, successive entries
// `step` bytes apart.  top is the LDS byte address of the next free entry.
typedef __attribute__((address_space(3))) int32_t lds_int;
struct LaneStack {
    uint32_t base, first, step;
    // stk: this lane's first entry; a wave's lanes own 64 consecutive columns or part of them,
    // so an address below `first` (scalar) is a first entry, whichever lane asks
    __device__ LaneStack(int32_t* stk, int stride)
        : base((uint32_t)(uintptr_t)(lds_int*)stk), step(4u * (uint32_t)stride)
    {
        first = (uint32_t)__builtin_amdgcn_readfirstlane((int)base) + 252u;
    }
    // an entry that stays only where keep: written in any case (the slot at top is free by
    // the stack bound), so no branch
    __device__ void push_if(uint32_t& top, int32_t r, bool keep) const
    {
        *(lds_int*)(uintptr_t)top = r;
        top += keep ? step : 0u;
    }
    __device__ int32_t pop(uint32_t& top) const
    {
        if (top <= first) return kDone;
        top -= step;
        return *(lds_int*)(uintptr_t)top;
    }
};

// Element i of an array.  Trees with the 32-entry stack keep every array below 4 GB
// (traversal_stack), so their loads take the array's scalar base plus a 32-bit offset,
// without 64-bit address arithmetic per load.
template <bool WIDE, class T> __device__ inline T load_at(const void* base, uint32_t i, uint32_t size, uint32_t off)
{
    if constexpr (WIDE) return *(const T*)((const char*)base + (size_t)i * size + off);
    else return *(const T*)((const char*)base + ((size == 48u ? (i + 2u * i) << 4 : i * size) + off));
}

typedef _Float16 half8 __attribute__((ext_vector_type(8), aligned(8)));

// (distance, child ref) pairs as one 64-bit float: the distance's bits are the high word, so
// the doubles order as the distances do (never a NaN: the high word is at most that of
// binary32 infinity, a finite double; binary64 keeps denormals) and v_min_f64 / v_max_f64,
// issued at the binary32 rate, move both words of a comparator in two instructions
// instead of a compare and four selects.
__device__ inline double pair(float k, int32_t r) { return __hiloint2double(__float_as_int(k), r); }
__device__ inline void pair_sort(double& a, double& b)
{
    double lo, hi;
    asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
    asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
    a = lo; b = hi;
}
__device__ inline bool pair_hit(double p) { return __int_as_float(__double2hiint(p)) < __builtin_huge_valf(); }

// max / min of three and of two without the quieting of signalling NaNs that fmaxf's
// lowering adds for values it cannot trace (box planes and distances are never one)
__device__ inline float vmax3(float a, float b, float c) { float r; asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c)); return r; }
__device__ inline float vmin3(float a, float b, float c) { float r; asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c)); return r; }
__device__ inline float vmax(float a, float b) { float r; asm("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b)); return r; }
__device__ inline float vmin(float a, float b) { float r; asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b)); return r; }

// what a ray's box tests need.  idir is the inverse direction divided by the nodes' scale, noi
// = -o * inverse direction: with c = origin * idir + noi per node and axis, a plane's
// distance along the ray is one fma, distance from the origin * idir + c.  That differs from
// (plane - o) * inverse direction by a few ulp of |o * inverse direction|, i.e. |o| * 2e-7 in
// distance, while every child box is inflated by DELTA_BSP = max|coordinate| * 1e-5: for origins up
// to 50 times the largest coordinate away culling is conservative, and the hit, decided only by
// the triangle test, is unchanged.  From farther away a ray that grazes a box may lose it, as it may with
// binary32 planes; their outward rounding makes that rarer.  55,000 to 44,000 hits at edges and
// corners of 600 triangles within [-1, 1]^3, lost from 1000 / 3000 / 10,000 away: binary32 planes
// 12 / 33 / 83, these 0 / 9 / 64, and none from 5 to 400.  near: byte offsets of the axes' near planes in a
// node, a byte each.
struct RayBox { float3 idir, noi; uint32_t near; };

__device__ inline float3 safe_inv(float3 d)
{
    float x = fabsf(d.x) < 1e-30f ? copysignf(1e-30f, d.x) : d.x;
    float y = fabsf(d.y) < 1e-30f ? copysignf(1e-30f, d.y) : d.y;
    float z = fabsf(d.z) < 1e-30f ? copysignf(1e-30f, d.z) : d.z;
    return make_float3(1.0f / x, 1.0f / y, 1.0f / z);
}

__device__ inline RayBox ray_box(const float3 o, const float3 d, float unscale)
{
    RayBox r;
    r.idir = safe_inv(d);
    r.noi = make_float3(-o.x * r.idir.x, -o.y * r.idir.y, -o.z * r.idir.z);
    r.idir.x *= unscale; r.idir.y *= unscale; r.idir.z *= unscale;
    // (by the inverse: -0 has a negative one)
    r.near = (r.idir.x < 0.f ? 8u : 0u) | (r.idir.y < 0.f ? 32u : 24u) << 8 | (r.idir.z < 0.f ? 72u : 64u) << 16;
    return r;
}

// One BVH4 node: the four child-box slab tests, then the children that are hit.  The
// nearest child is returned as the next ref, the others go on the stack farthest first
// (ORDERED; else any order).  No child hit: the next ref is popped.  The tree is collapsed
// so that the stack never holds more than STACK-1 entries.
//
// Per axis one load brings the near planes (lo or hi by the direction's sign), then the far
// ones: near <= far (fma is monotonic), so entry and exit are a max3 / min3 of three fmas
// per child without a min/max pair per axis.
//
// Bound by VALU issue.  SQ and TA counters of a 1024-ray gather over 50k triangles (751k
// texels), seven binary32 loads a visit -> these five binary16 ones: time 84.9 -> 71.0 ms, VALU
// 78% -> 94% of issue, L1 tag lookups (one per distinct node and load) 46.7e9 -> 35.1e9, TA
// busy 86% -> 79%; sun-and-sky bake over 132k triangles 24.2 -> 22.3 ms.  1M random rays
// against 100k triangles, bound by latency at 20% active lanes, stayed at 0.638 ms (0.49 now, by their
// launch shape).
// Straight-line tests, pairs sorted as doubles, branch-free pushes and 32-bit offsets had
// taken the gather's wave instructions from 49.7e9 to 39.7e9 (89.6 -> 84.9 ms).
template <bool WIDE, bool ORDERED>
__device__ inline int32_t visit4(const NodeT* __restrict__ nodes, int32_t ref, const RayBox& R, float tlo, float thi,
                                 const LaneStack& stk, uint32_t& top)
{
    const uint32_t n = (uint32_t)ref;
    // the node's five 16-byte loads are issued together, before any use (left to itself the
    // scheduler issues some, waits for them, then the others)
    const half8 x = load_at<WIDE, half8>(nodes, n, 128u, R.near & 255u), y = load_at<WIDE, half8>(nodes, n, 128u, (R.near >> 8) & 255u);
    const half8 z = load_at<WIDE, half8>(nodes, n, 128u, R.near >> 16);
    const float4 org = load_at<WIDE, float4>(nodes, n, 128u, 96u);
    const int4 r = load_at<WIDE, int4>(nodes, n, 128u, 48u);
    __builtin_amdgcn_sched_barrier(0);
    const float cx = __fmaf_rn(org.x, R.idir.x, R.noi.x), cy = __fmaf_rn(org.y, R.idir.y, R.noi.y), cz = __fmaf_rn(org.z, R.idir.z, R.noi.z);
    auto enter = [&](int k) {
        return vmax3(__fmaf_rn((float)x[k], R.idir.x, cx), __fmaf_rn((float)y[k], R.idir.y, cy), vmax(__fmaf_rn((float)z[k], R.idir.z, cz), tlo));
    };
    auto leave = [&](int k) {
        return vmin3(__fmaf_rn((float)x[4 + k], R.idir.x, cx), __fmaf_rn((float)y[4 + k], R.idir.y, cy),
                     vmin(__fmaf_rn((float)z[4 + k], R.idir.z, cz), thi));
    };
    const float k0 = enter(0), k1 = enter(1), k2 = enter(2), k3 = enter(3);
    // (bitwise, so that the tests stay straight-line code)
    const bool h0 = (r.x != kNoChild) & (k0 <= leave(0)), h1 = (r.y != kNoChild) & (k1 <= leave(1));
    const bool h2 = (r.z != kNoChild) & (k2 <= leave(2)), h3 = (r.w != kNoChild) & (k3 <= leave(3));
    if constexpr (!ORDERED) {
        // any order: continue with the last hit child in slot order, push the others
        int32_t nxt = h0 ? r.x : kDone;
        stk.push_if(top, nxt, h1 & h0);
        bool have = h0 | h1;
        nxt = h1 ? r.y : nxt;
        stk.push_if(top, nxt, h2 & have);
        have = have | h2;
        nxt = h2 ? r.z : nxt;
        stk.push_if(top, nxt, h3 & have);
        nxt = h3 ? r.w : nxt;
        return nxt != kDone ? nxt : stk.pop(top);
    }
    constexpr float kInf = __builtin_huge_valf();
    double p0 = pair(h0 ? k0 : kInf, r.x), p1 = pair(h1 ? k1 : kInf, r.y), p2 = pair(h2 ? k2 : kInf, r.z), p3 = pair(h3 ? k3 : kInf, r.w);
    pair_sort(p0, p1); pair_sort(p2, p3); pair_sort(p0, p2); pair_sort(p1, p3); pair_sort(p1, p2);
    stk.push_if(top, __double2loint(p3), pair_hit(p3));
    stk.push_if(top, __double2loint(p2), pair_hit(p2));
    stk.push_if(top, __double2loint(p1), pair_hit(p1));
    return pair_hit(p0) ? __double2loint(p0) : stk.pop(top);
}

// Closest accepted hit of one ray, resumable: trace_begin sets a ray up, trace_resume runs
// it until it is finished (returns true) or until no more than `yield_at` lanes of the
// wave are still tracing (returns false, state kept), trace_finish gives its hit.  The
// state keeps the best hit's leaf-order slot and distance; triangle, side and hitPoint2d
// are recomputed from the slot's record once per ray, bit-identical to the test's.
struct TraceState {
    float3 o, d;
    RayBox box;
    float lo, best, bound;
    int32_t ref, leaf;
    uint32_t slot, top;
};

// false when the ray misses the scene box (then it is finished, no hit)
__device__ inline bool trace_begin(TraceState& S, const ColliderView& c, const float3 o, const float3 d, float rmin, float rmax,
                                   const LaneStack& stk)
{
    float lo, hi;
    S.slot = kNoSlot;
    if (!c.nvalid || !ref_box_intersect(c.bmin, c.bmax, o, d, rmin, rmax, lo, hi)) return false;
    S.o = o; S.d = d;
    S.box = ray_box(o, d, c.unscale);
    S.lo = lo; S.best = hi; S.bound = hi;
    S.ref = c.root4; S.leaf = 0; S.top = stk.base;
    return true;
}

// One triangle against the ray: slot p with plane pl and record (sv, ev, mt) (all zero where
// the caller has not read it: LATE reads it here, once the plane test passes).  True when it
// is an accepted hit that ends the search (the ray's state alone does not tell: S.ref is kDone
// on every ray's last leaf too, and S.best starts as the clipped range).
template <bool WIDE, bool LATE, class Filter>
__device__ inline bool test_triangle(TraceState& S, const Filter& flt, const ColliderView& c, uint32_t p, const float4 pl, float4 sv,
                                     float4 ev, uint4 mt)
{
    float ndd;
    const float t = plane_distance(pl, S.o, S.d, ndd);
    if (!(t >= S.lo && t <= S.bound)) return false;
    if constexpr (LATE) {
        // the whole record in one round trip
        sv = load_at<WIDE, float4>(c.rest, p, 48u, 0u); ev = load_at<WIDE, float4>(c.rest, p, 48u, 16u);
        mt = load_at<WIDE, uint4>(c.rest, p, 48u, 32u);
        __builtin_amdgcn_sched_barrier(0);
    }
    float u, v;
    if (!srlnp_hit(sv, ev, mt.z, S.o, S.d, t, u, v)) return false;
    // a tie goes to the lower triangle index
    if (t == S.best && S.slot != kNoSlot && mt.x >= load_at<WIDE, uint32_t>(c.rest, S.slot, 48u, 32u)) return false;
    if (!flt.accept(mt.x, ndd < 0, t, u, v)) return false;
    S.best = t; S.slot = p;
    S.bound = flt.clamp(t);
    if (!flt.done(t)) return false;
    S.ref = kDone;
    return true;
}

// Loop shape: "while-while" with speculative traversal (Aila & Laine, HPG 2009).
// Lanes descend inner nodes; a lane that reaches a leaf parks it and keeps
// descending, until every lane of the wave holds a parked leaf; then the wave tests
// triangles together.  Inner-node and triangle work thus run with full lane masks
// instead of interleaving per iteration.  The result does not depend on the visiting
// order (see the header), so it is the same as any other order's.
// ORDERED = false (shadow rays): children are visited in any order.  A shadow ray only
// asks whether a blocker lies below rugDistance and, if not, whether any blocker lies in
// range; after the first hit its range shrinks below rugDistance and the search there is
// exhaustive, so the answer does not depend on the order, and the sort is saved.
// EAGER (scattered rays, bound by latency): a leaf's triangles are read two at a time with
// plane and record together, one memory round trip instead of four.
template <int STACK, bool STATS, class Filter, bool ORDERED, bool YIELD, bool EAGER>
__device__ inline bool trace_run(TraceState& S, const Filter& flt, const ColliderView& c, const LaneStack& stk, uint32_t yield_at,
                                 uint32_t& nvis, uint32_t& ntest)
{
    constexpr bool WIDE = STACK > 32;
    while (S.ref != kDone || S.leaf < 0) {
        if (YIELD && (uint32_t)__popcll(__ballot(1)) <= yield_at) return false;     // enough lanes are free
        // inner nodes, parking the first leaf met
        while (S.ref >= 0 && S.ref != kDone) {
            if (STATS) nvis++;
            S.ref = visit4<WIDE, ORDERED>(c.nodes4, S.ref, S.box, S.lo, S.bound, stk, S.top);
            if (S.ref < 0 && S.leaf == 0) { S.leaf = S.ref; S.ref = stk.pop(S.top); }
            if (!__any(S.leaf == 0)) break;              // every active lane holds a leaf
        }
        // a leaf reached outside the loop above (the root itself, or a leaf next on
        // the stack while none was parked) is parked here, so every pass progresses
        if (S.leaf == 0 && S.ref < 0) { S.leaf = S.ref; S.ref = stk.pop(S.top); }
        // triangles of the parked leaf, then of leaves met directly on the stack
        while (S.leaf < 0) {
            const uint32_t st = leaf_start(S.leaf), end = st + leaf_count(S.leaf);
            S.leaf = 0;
            const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
            if constexpr (EAGER) {
                for (uint32_t p = st; p < end; p += 2) {
                    const uint32_t q = min(p + 1, end - 1);
                    const float4 pl0 = load_at<WIDE, float4>(c.plane, p, 16u, 0u), pl1 = load_at<WIDE, float4>(c.plane, q, 16u, 0u);
                    const float4 sv0 = load_at<WIDE, float4>(c.rest, p, 48u, 0u), ev0 = load_at<WIDE, float4>(c.rest, p, 48u, 16u);
                    const float4 sv1 = load_at<WIDE, float4>(c.rest, q, 48u, 0u), ev1 = load_at<WIDE, float4>(c.rest, q, 48u, 16u);
                    const uint4 mt0 = load_at<WIDE, uint4>(c.rest, p, 48u, 32u), mt1 = load_at<WIDE, uint4>(c.rest, q, 48u, 32u);
                    __builtin_amdgcn_sched_barrier(0);
                    if (STATS) ntest += q - p + 1;
                    if (test_triangle<WIDE, false>(S, flt, c, p, pl0, sv0, ev0, mt0)) break;
                    if (q != p && test_triangle<WIDE, false>(S, flt, c, q, pl1, sv1, ev1, mt1)) break;
                }
            } else {
                for (uint32_t p = st; p < end; p++) {
                    if (STATS) ntest++;
                    if (test_triangle<WIDE, true>(S, flt, c, p, load_at<WIDE, float4>(c.plane, p, 16u, 0u), zero, zero, make_uint4(0u, 0u, 0u, 0u))) break;
                }
            }
            if (S.ref < 0) { S.leaf = S.ref; S.ref = stk.pop(S.top); }
        }
    }
    return true;
}

template <int STACK, bool EAGER, class Filter>
__device__ inline bool trace_resume(TraceState& S, const Filter& flt, const ColliderView& c, const LaneStack& stk, uint32_t yield_at)
{
    uint32_t a = 0, b = 0;
    return trace_run<STACK, false, Filter, true, true, EAGER>(S, flt, c, stk, yield_at, a, b);
}

// the hit of a finished ray (tri -1: none)
__device__ inline void trace_finish(const TraceState& S, const ColliderView& c, TraceResult& res)
{
    res.tri = -1; res.slot = S.slot;
    if (S.slot == kNoSlot) return;
    const float4 pl = c.plane[S.slot];
    const TriRest* tr = c.rest + S.slot;
    res.tri = (int)tr->meta.x;
    res.t = S.best;
    res.front = S.d.x * pl.x + S.d.y * pl.y + S.d.z * pl.z < 0;
    srlnp_hit(tr->sv, tr->ev, tr->axes, S.o, S.d, S.best, res.u, res.v);
}

// the whole ray at once
template <int STACK, bool STATS, class Filter, bool ORDERED = true, bool EAGER = false>
__device__ inline void trace_closest(const Filter& flt, const ColliderView& c, const float3 o, const float3 d, float rmin, float rmax,
                                     int32_t* stk, int stride, TraceResult& res, uint32_t& nvis, uint32_t& ntest)
{
    TraceState S;
    const LaneStack ls(stk, stride);
    res.tri = -1;
    if (!trace_begin(S, c, o, d, rmin, rmax, ls)) return;
    trace_run<STACK, STATS, Filter, ORDERED, false, EAGER>(S, flt, c, ls, 0u, nvis, ntest);
    trace_finish(S, c, res);
}

} // namespace lsg
