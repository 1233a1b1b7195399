// lsgpu_sah.hip -- SAH rebuild of the LBVH's inner nodes on the GPU.
//
// The same tree as the host rebuild (lsgpu_sah.cpp, lsg_bvh_rebuild_sah), built breadth
// first: the leaves of the LBVH (triangle ranges of at most leaf_size, in the order of their
// triangles) are rebuilt top-down, one wave per node of a level (16 waves from kMidTask leaves
// on).  It bins its leaves' centroids (32 bins per axis, as many as leaves below 32) into LDS, a
// wave picks the cheapest split as the host does (area(left)·n(left) + area(right)·n(right) over
// the three axes; equal centroids split the range in half), and the leaves are partitioned
// stably into the other buffer, collecting the children's boxes and centroid bounds.  Box and bound
// reductions are exact (min/max over floats as order-preserving integers), the split
// arithmetic is the host's, and nodes are numbered in preorder (left child = node + 1, right
// child = node + leaves on the left), so the result equals the host's node for node.
// Tasks of 2^15 leaves or more (the top levels) take the same steps across the chip:
// many workgroups bin, one wave splits, a scan of left/right flags partitions.
//
// The levels are short and depend on one another, so what a level costs is its slowest node and
// the host's look at the next level's size.  50,000 triangles: 18 levels of 150 us (one lane
// walking 3 x 32 bins twice, one wave over the root's 25,000 leaves) -> 94 us for the seven with
// large nodes and 32 us below them, the collider's build 4.5 ms -> 3.1 ms.
#include "lsgpu_internal.h"
#include <algorithm>
#include <cmath>
#include <vector>

namespace lsg {
namespace {

constexpr int kSahBins = 32;

struct SahLeaf { int32_t ref; float b[6]; float c[3]; };
struct SahTask { uint32_t begin, end, id, depth; float clo[3], chi[3]; };
struct SahLevel { uint32_t ntask, maxm; };         // a level's tasks and the most leaves of one

// floats as integers of the same order (-0 as +0), for atomic min/max
__device__ inline int f2o(float x)
{
    int i = __float_as_int(x);
    if (i == (int)0x80000000) i = 0;
    return i >= 0 ? i : (i ^ 0x7fffffff);
}
__device__ inline float o2f(int i) { return __int_as_float(i >= 0 ? i : (i ^ 0x7fffffff)); }

__device__ inline bool reachable(int i, const int* first, const int* last, uint32_t leafmax)
{
    return (uint32_t)(last[i] - first[i] + 1) > leafmax;   // the root has every triangle
}

// leaves of the LBVH: each reachable node's children of at most leafmax triangles
__global__ __launch_bounds__(256) void k_sah_mark(int ni, const int* __restrict__ first, const int* __restrict__ last,
                                                  const int* __restrict__ split, uint32_t leafmax, uint32_t* __restrict__ flag)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= ni || !reachable(i, first, last, leafmax)) return;
    const int g = split[i];
    if ((uint32_t)(g - first[i] + 1) <= leafmax) flag[first[i]] = 1u;
    if ((uint32_t)(last[i] - g) <= leafmax) flag[g + 1] = 1u;
}

__global__ __launch_bounds__(256) void k_sah_gather(int ni, const int* __restrict__ first, const int* __restrict__ last,
                                                    const int* __restrict__ split, uint32_t leafmax, const Node* __restrict__ nodes,
                                                    const uint32_t* __restrict__ pos, SahLeaf* __restrict__ L)
{
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= ni || !reachable(i, first, last, leafmax)) return;
    const int g = split[i];
    const Node q = nodes[i];
    const float f[16] = {q.q0.x, q.q0.y, q.q0.z, q.q0.w, q.q1.x, q.q1.y, q.q1.z, q.q1.w,
                         q.q2.x, q.q2.y, q.q2.z, q.q2.w, q.q3.x, q.q3.y, q.q3.z, q.q3.w};
    for (int c = 0; c < 2; c++) {
        const int cf = c == 0 ? first[i] : g + 1;
        const int cl = c == 0 ? g : last[i];
        if ((uint32_t)(cl - cf + 1) > leafmax) continue;
        SahLeaf lf;
        lf.ref = __float_as_int(f[12 + c]);
        for (int k = 0; k < 6; k++) lf.b[k] = f[6 * c + k];
        for (int a = 0; a < 3; a++) lf.c[a] = (lf.b[2 * a] + lf.b[2 * a + 1]) * 0.5f;
        L[pos[cf]] = lf;
    }
}

// centroid bounds of all leaves (the root task's), as ordered integers: lo x y z, hi x y z
__global__ __launch_bounds__(256) void k_sah_root(const SahLeaf* __restrict__ L, uint32_t n, int* __restrict__ cb)
{
    __shared__ int s[6];
    if (threadIdx.x < 6) s[threadIdx.x] = threadIdx.x < 3 ? f2o(3.0e38f) : f2o(-3.0e38f);
    __syncthreads();
    for (uint32_t k = blockIdx.x * 256 + threadIdx.x; k < n; k += gridDim.x * 256) {
        for (int a = 0; a < 3; a++) {
            atomicMin(&s[a], f2o(L[k].c[a]));
            atomicMax(&s[3 + a], f2o(L[k].c[a]));
        }
    }
    __syncthreads();
    if (threadIdx.x < 3) atomicMin(&cb[threadIdx.x], s[threadIdx.x]);
    else if (threadIdx.x < 6) atomicMax(&cb[threadIdx.x], s[threadIdx.x]);
}

__global__ void k_sah_root_task(const int* __restrict__ cb, uint32_t n, SahTask* __restrict__ t, SahLevel* __restrict__ lev)
{
    if (threadIdx.x) return;
    lev->ntask = 1; lev->maxm = n;
    SahTask r;
    r.begin = 0; r.end = n; r.id = 0; r.depth = 1;
    for (int a = 0; a < 3; a++) { r.clo[a] = o2f(cb[a]); r.chi[a] = o2f(cb[3 + a]); }
    *t = r;
}

// bins per axis of a task and the binning scale (0 on an axis whose centroids coincide)
__device__ inline int task_bins(const SahTask& T, bool* ok, float* sc)
{
    const uint32_t m = T.end - T.begin;
    const int nb = (int)min((uint32_t)kSahBins, max(4u, m));
    for (int a = 0; a < 3; a++) {
        ok[a] = T.chi[a] > T.clo[a];
        sc[a] = ok[a] ? (float)nb / (T.chi[a] - T.clo[a]) : 0.f;
    }
    return nb;
}

__device__ inline int bin_of(const SahLeaf& f, const SahTask& T, int a, float sc, int nb)
{
    return min((int)((f.c[a] - T.clo[a]) * sc), nb - 1);
}

struct SahSweep { uint32_t c; float b[6]; };

__device__ inline void sweep_add(SahSweep& a, bool on, int lane_delta)
{
    // the bins of another lane of this half wave added to this lane's, in range
    SahSweep o;
    o.c = lane_delta < 0 ? (uint32_t)__shfl_up((int)a.c, -lane_delta, 32) : (uint32_t)__shfl_down((int)a.c, lane_delta, 32);
    for (int e = 0; e < 6; e++) {
        o.b[e] = lane_delta < 0 ? __shfl_up(a.b[e], -lane_delta, 32) : __shfl_down(a.b[e], lane_delta, 32);
        if (on) a.b[e] = (e & 1) ? fmaxf(a.b[e], o.b[e]) : fminf(a.b[e], o.b[e]);
    }
    if (on) a.c += o.c;
}

__device__ inline float sweep_area(const SahSweep& s)
{
    const float dx = s.b[1] - s.b[0], dy = s.b[3] - s.b[2], dz = s.b[5] - s.b[4];
    return dx * dy + dy * dz + dz * dx;
}

// The host's split search (lsgpu_sah.cpp) on a task's bins: dec = (axis or -1 for halves, last
// bin on the left, leaves on the left).  One wave: a lane per (axis, bin), axes 0 and 1 in the
// half waves, then axis 2.  Boxes and counts of the bins up to a lane's and after it come from
// scans (minima and maxima are exact in any order), every split's cost is the host's
// expression, and of equal costs the first in the host's order is taken.  A NaN cost is never
// below another, so it is taken only where the host meets it first.
__device__ inline void sah_choose(const int (*cnt)[kSahBins], const int (*box)[kSahBins][6], int nb, const bool* ok, uint32_t m,
                                  int* dec)
{
    const uint32_t lane = threadIdx.x & 63u;
    const int k = (int)(lane & 31u);
    uint64_t best = ~0ull;                       // (ordered cost, axis, bin)
    uint32_t first = ~0u;                        // (axis, bin, NaN) of the first split
    uint32_t left[2];
    for (int pass = 0; pass < 2; pass++) {
        const int a = pass ? 2 : (int)(lane >> 5);
        const bool have = (pass == 0 || lane < 32) && k < nb;
        SahSweep s{0u, {3.0e38f, -3.0e38f, 3.0e38f, -3.0e38f, 3.0e38f, -3.0e38f}};
        if (have) {
            s.c = (uint32_t)cnt[a][k];
            for (int e = 0; e < 6; e++) s.b[e] = o2f(box[a][k][e]);
        }
        SahSweep r = s;
        for (int d = 1; d < 32; d <<= 1) {
            sweep_add(s, k >= d, -d);
            sweep_add(r, k + d < 32, d);
        }
        left[pass] = s.c;
        const float ra = __shfl_down(r.c ? sweep_area(r) : 0.f, 1, 32);
        const uint32_t rc = (uint32_t)__shfl_down((int)r.c, 1, 32);
        const bool okay = a == 0 ? ok[0] : (a == 1 ? ok[1] : ok[2]);
        if (have && okay && k < nb - 1 && s.c && rc) {
            const float cost = sweep_area(s) * (float)s.c + ra * (float)rc;
            const uint32_t at = (uint32_t)(a * 32 + k);
            const bool nan = cost != cost;
            first = min(first, at * 2u + (nan ? 1u : 0u));
            if (!nan) best = min(best, (uint64_t)((uint32_t)f2o(cost) ^ 0x80000000u) << 32 | at);
        }
    }
    for (int o = 32; o; o >>= 1) {
        first = min(first, (uint32_t)__shfl_xor((int)first, o));
        const uint64_t b = (uint64_t)(uint32_t)__shfl_xor((int)(uint32_t)best, o) | (uint64_t)(uint32_t)__shfl_xor((int)(uint32_t)(best >> 32), o) << 32;
        best = min(best, b);
    }
    int bax = -1, bk = -1;
    uint32_t nl = m / 2;
    if (first != ~0u) {
        const uint32_t at = (first & 1u) ? first >> 1 : (uint32_t)best;
        bax = (int)(at >> 5); bk = (int)(at & 31u);
        nl = (uint32_t)__shfl((int)(bax == 2 ? left[1] : left[0]), bax == 1 ? 32 + bk : bk);
    }
    if (lane == 0) { dec[0] = bax; dec[1] = bk; dec[2] = (int)nl; }
}

// a split task's node (children's boxes, a leaf child's ref from dst) and its children of
// two or more leaves as the next level's tasks
__device__ inline void sah_emit(const SahTask& T, uint32_t nl, const int (*child)[12], const SahLeaf* dst, Node* out, SahTask* next,
                                SahLevel* nlev, uint32_t* depth)
{
    atomicMax(depth, T.depth);
    float nodef[16];
    // the children of two or more leaves become tasks, appended with one atomic
    const uint32_t nkids = (nl >= 2 ? 1u : 0u) + (T.end - T.begin - nl >= 2 ? 1u : 0u);
    uint32_t slot = nkids ? atomicAdd(&nlev->ntask, nkids) : 0u;
    if (nkids) atomicMax(&nlev->maxm, max(nl, T.end - T.begin - nl));
    for (int s = 0; s < 2; s++) {
        const uint32_t b = s == 0 ? T.begin : T.begin + nl, e = s == 0 ? T.begin + nl : T.end;
        const uint32_t ms = e - b;
        const uint32_t id = s == 0 ? T.id + 1 : T.id + nl;
        const int32_t ref = ms == 1 ? dst[b].ref : (int32_t)id;
        for (int k = 0; k < 6; k++) nodef[6 * s + k] = o2f(child[s][k]);
        nodef[12 + s] = __int_as_float(ref);
        if (ms >= 2) {
            SahTask c;
            c.begin = b; c.end = e; c.id = id; c.depth = T.depth + 1;
            for (int a = 0; a < 3; a++) { c.clo[a] = o2f(child[s][6 + a]); c.chi[a] = o2f(child[s][9 + a]); }
            next[slot++] = c;
        }
    }
    nodef[14] = 0.f; nodef[15] = 0.f;
    Node nd;
    nd.q0 = make_float4(nodef[0], nodef[1], nodef[2], nodef[3]);
    nd.q1 = make_float4(nodef[4], nodef[5], nodef[6], nodef[7]);
    nd.q2 = make_float4(nodef[8], nodef[9], nodef[10], nodef[11]);
    nd.q3 = make_float4(nodef[12], nodef[13], nodef[14], nodef[15]);
    out[T.id] = nd;
}

__device__ inline void bins_init(int* cnt, int* box, uint32_t tid, uint32_t nthreads)
{
    const int kLo = f2o(3.0e38f), kHi = f2o(-3.0e38f);
    for (uint32_t k = tid; k < 3 * kSahBins; k += nthreads) {
        cnt[k] = 0;
        for (int e = 0; e < 6; e++) box[6 * k + e] = (e & 1) ? kHi : kLo;
    }
}

// per child: box lo/hi x y z (6), centroid lo x y z, hi x y z (6)
__device__ constexpr bool child_high(int e) { return e < 6 ? (e & 1) != 0 : e >= 9; }

__device__ inline void child_init(int* child, uint32_t tid)
{
    if (tid < 24) child[tid] = child_high((int)(tid % 12)) ? f2o(-3.0e38f) : f2o(3.0e38f);
}

__device__ inline void bin_leaf(const SahLeaf& f, const SahTask& T, const bool* ok, const float* sc, int nb, int (*cnt)[kSahBins],
                                int (*box)[kSahBins][6])
{
    for (int a = 0; a < 3; a++) {
        if (!ok[a]) continue;
        const int j = bin_of(f, T, a, sc[a], nb);
        atomicAdd(&cnt[a][j], 1);
        for (int e = 0; e < 6; e++) {
            if (e & 1) atomicMax(&box[a][j][e], f2o(f.b[e]));
            else atomicMin(&box[a][j][e], f2o(f.b[e]));
        }
    }
}

__device__ inline void child_add(int* cbx, const SahLeaf& f)
{
    for (int e = 0; e < 6; e++) {
        if (e & 1) atomicMax(&cbx[e], f2o(f.b[e]));
        else atomicMin(&cbx[e], f2o(f.b[e]));
    }
    for (int a = 0; a < 3; a++) {
        atomicMin(&cbx[6 + a], f2o(f.c[a]));
        atomicMax(&cbx[9 + a], f2o(f.c[a]));
    }
}

// the smaller (larger) of v over the 16 lanes of a row, in every lane of it
template <bool MAX> __device__ inline int row_extreme(int v)
{
    auto pick = [](int a, int b) { return MAX ? max(a, b) : min(a, b); };
    v = pick(v, __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, true));      // lane ^ 1
    v = pick(v, __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, true));      // lane ^ 2
    v = pick(v, __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, true));     // mirrored in 8
    v = pick(v, __builtin_amdgcn_update_dpp(0, v, 0x140, 0xf, 0xf, true));     // mirrored in 16
    return v;
}

// the nodes of a level of lo to hi - 1 leaves, one per workgroup of TH lanes: bins, split, stable
// partition src -> dst, children.  The children's boxes and centroid bounds are kept per lane and
// reduced once (all lanes of a wave adding to one LDS word would serialise).
template <int TH>
__global__ __launch_bounds__(TH) void k_sah_level(const SahTask* __restrict__ tasks, const SahLevel* __restrict__ lev, uint32_t lo, uint32_t hi,
                                                  const SahLeaf* __restrict__ src, SahLeaf* __restrict__ dst, Node* __restrict__ out,
                                                  SahTask* __restrict__ next, SahLevel* __restrict__ nlev, uint32_t* __restrict__ depth)
{
    __shared__ int s_cnt[3][kSahBins];
    __shared__ int s_box[3][kSahBins][6];
    __shared__ int s_child[2][12];
    __shared__ int s_dec[3];                // axis (-1: halves), bin, leaves on the left
    __shared__ uint32_t s_left[TH / 64];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t ntask = lev->ntask;
    for (uint32_t q = blockIdx.x; q < ntask; q += gridDim.x) {
        const SahTask T = tasks[q];
        const uint32_t m = T.end - T.begin;
        if (m < lo || m >= hi) continue;
        bool ok[3];
        float sc[3];
        const int nb = task_bins(T, ok, sc);
        bins_init(&s_cnt[0][0], &s_box[0][0][0], tid, TH);
        child_init(&s_child[0][0], tid);
        __syncthreads();
        for (uint32_t k = T.begin + tid; k < T.end; k += TH) bin_leaf(src[k], T, ok, sc, nb, s_cnt, s_box);
        __syncthreads();
        if (wave == 0) sah_choose(s_cnt, s_box, nb, ok, m, s_dec);
        __syncthreads();
        const int bax = s_dec[0], bk = s_dec[1];
        const uint32_t nl = (uint32_t)s_dec[2];
        const float clo = bax == 0 ? T.clo[0] : (bax == 1 ? T.clo[1] : T.clo[2]), scb = bax == 0 ? sc[0] : (bax == 1 ? sc[1] : sc[2]);
        uint32_t ldone = 0;
        int ext[2][12];
        for (int c = 0; c < 2; c++)
            for (int e = 0; e < 12; e++) ext[c][e] = child_high(e) ? f2o(-3.0e38f) : f2o(3.0e38f);
        for (uint32_t base = T.begin; base < T.end; base += TH) {
            const uint32_t k = base + tid;
            const bool valid = k < T.end;
            SahLeaf f;
            bool left = false;
            if (valid) {
                f = src[k];
                const float c = bax == 0 ? f.c[0] : (bax == 1 ? f.c[1] : f.c[2]);
                left = bax < 0 ? (k - T.begin < m / 2) : (min((int)((c - clo) * scb), nb - 1) <= bk);      // bin_of on that axis
            }
            const uint64_t lm = __ballot(valid && left);
            uint32_t before = ldone, all = (uint32_t)__popcll(lm);
            if (TH > 64) {
                if (lane == 0) s_left[wave] = all;
                __syncthreads();
                all = 0;
                for (uint32_t w = 0; w < TH / 64; w++) {
                    if (w < wave) before += s_left[w];
                    all += s_left[w];
                }
                __syncthreads();
            }
            before += (uint32_t)__popcll(lm & ((1ull << lane) - 1ull));     // leaves on the left before this one
            if (valid) {
                dst[left ? T.begin + before : T.begin + nl + (k - T.begin - before)] = f;
                int v[12];
                for (int e = 0; e < 6; e++) v[e] = f2o(f.b[e]);
                for (int a = 0; a < 3; a++) v[6 + a] = v[9 + a] = f2o(f.c[a]);
                for (int c = 0; c < 2; c++)
                    if (left == (c == 0))
                        for (int e = 0; e < 12; e++) ext[c][e] = child_high(e) ? max(ext[c][e], v[e]) : min(ext[c][e], v[e]);
            }
            ldone += all;
        }
        for (int c = 0; c < 2; c++)
            for (int e = 0; e < 12; e++) {
                const int v = child_high(e) ? row_extreme<true>(ext[c][e]) : row_extreme<false>(ext[c][e]);
                if ((lane & 15u) == 0) { if (child_high(e)) atomicMax(&s_child[c][e], v); else atomicMin(&s_child[c][e], v); }
            }
        __syncthreads();
        if (tid == 0) sah_emit(T, nl, s_child, dst, out, next, nlev, depth);
        __syncthreads();
    }
}

// ---- one big task across the chip ------------------------------------------------------
// The top levels have a handful of tasks over millions of leaves: each is binned by many
// workgroups (LDS bins merged into global ones with the same exact integer min/max and
// counts), split by one wave with the same search, partitioned stably by a scan of its
// left/right flags, and emitted as k_sah_level emits.
constexpr uint32_t kBigTask = 1u << 15;
// from here on a task has 16 waves (the build of 50,000 triangles takes 3.03 to 3.16 ms with the
// line anywhere from 2^7 to 2^11; one wave for all: 4.5 ms)
constexpr uint32_t kMidTask = 1u << 9;

struct SahBig {
    int cnt[3][kSahBins];
    int box[3][kSahBins][6];
    int child[2][12];
    int dec[3];
};

__global__ __launch_bounds__(256) void k_big_init(SahBig* __restrict__ B)
{
    bins_init(&B->cnt[0][0], &B->box[0][0][0], threadIdx.x, 256);
    child_init(&B->child[0][0], threadIdx.x);
}

__global__ __launch_bounds__(256) void k_big_bin(const SahTask* __restrict__ task, const SahLeaf* __restrict__ src, SahBig* __restrict__ B)
{
    __shared__ int s_cnt[3][kSahBins];
    __shared__ int s_box[3][kSahBins][6];
    const SahTask T = *task;
    bool ok[3];
    float sc[3];
    const int nb = task_bins(T, ok, sc);
    bins_init(&s_cnt[0][0], &s_box[0][0][0], threadIdx.x, 256);
    __syncthreads();
    for (uint32_t k = T.begin + blockIdx.x * 256 + threadIdx.x; k < T.end; k += gridDim.x * 256) bin_leaf(src[k], T, ok, sc, nb, s_cnt, s_box);
    __syncthreads();
    for (uint32_t k = threadIdx.x; k < 3 * kSahBins; k += 256) {
        const int c = (&s_cnt[0][0])[k];
        if (!c) continue;
        atomicAdd(&B->cnt[0][0] + k, c);
        for (int e = 0; e < 6; e++) {
            int* g = &B->box[0][0][0] + 6 * k + e;
            const int v = (&s_box[0][0][0])[6 * k + e];
            if (e & 1) atomicMax(g, v); else atomicMin(g, v);
        }
    }
}

__global__ __launch_bounds__(64) void k_big_split(const SahTask* __restrict__ task, SahBig* __restrict__ B)
{
    const SahTask T = *task;
    bool ok[3];
    float sc[3];
    const int nb = task_bins(T, ok, sc);
    sah_choose(B->cnt, B->box, nb, ok, T.end - T.begin, B->dec);
}

__global__ __launch_bounds__(256) void k_big_flag(const SahTask* __restrict__ task, const SahLeaf* __restrict__ src,
                                                  const SahBig* __restrict__ B, uint32_t* __restrict__ flag)
{
    const SahTask T = *task;
    const uint32_t m = T.end - T.begin;
    bool ok[3];
    float sc[3];
    const int nb = task_bins(T, ok, sc);
    const int bax = B->dec[0], bk = B->dec[1];
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < m; i += gridDim.x * 256)
        flag[i] = (bax < 0 ? i < m / 2 : bin_of(src[T.begin + i], T, bax, sc[bax], nb) <= bk) ? 1u : 0u;
}

__global__ __launch_bounds__(256) void k_big_scatter(const SahTask* __restrict__ task, const SahLeaf* __restrict__ src,
                                                     SahLeaf* __restrict__ dst, const uint32_t* __restrict__ flag,
                                                     const uint32_t* __restrict__ prefix, SahBig* __restrict__ B)
{
    __shared__ int s_child[2][12];
    const SahTask T = *task;
    const uint32_t m = T.end - T.begin, nl = (uint32_t)B->dec[2];
    child_init(&s_child[0][0], threadIdx.x);
    __syncthreads();
    for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < m; i += gridDim.x * 256) {
        const SahLeaf f = src[T.begin + i];
        const bool left = flag[i] != 0;
        dst[left ? T.begin + prefix[i] : T.begin + nl + (i - prefix[i])] = f;
        child_add(s_child[left ? 0 : 1], f);
    }
    __syncthreads();
    if (threadIdx.x < 24) {
        const uint32_t k = threadIdx.x, e = k % 12;
        int* g = &B->child[0][0] + k;
        const int v = (&s_child[0][0])[k];
        if (child_high((int)e)) atomicMax(g, v); else atomicMin(g, v);
    }
}

__global__ void k_big_emit(const SahTask* __restrict__ task, const SahLeaf* __restrict__ dst, const SahBig* __restrict__ B,
                           Node* __restrict__ out, SahTask* __restrict__ next, SahLevel* __restrict__ nlev, uint32_t* __restrict__ depth)
{
    if (threadIdx.x) return;
    sah_emit(*task, (uint32_t)B->dec[2], B->child, dst, out, next, nlev, depth);
}

// ---- BVH2 -> BVH4 collapse ------------------------------------------------------------

struct C4Work { int32_t i2; uint32_t slot, P; };

// heights (inner nodes on the longest path down, a node over two leaves = 1), one level
// per launch: launch k finishes the nodes whose inner children were finished by earlier
// launches (H in 1..k-1), so H = k is the height, and every box of H read was written
// before the launch began (no fences)
__global__ __launch_bounds__(256) void k_c4_height(uint32_t nn, const Node* __restrict__ nodes, uint32_t* __restrict__ H, uint32_t k)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nn || H[i]) return;
    const int32_t r0 = __float_as_int(nodes[i].q3.x), r1 = __float_as_int(nodes[i].q3.y);
    if (r0 >= 0) { const uint32_t h = H[r0]; if (h == 0 || h >= k) return; }
    if (r1 >= 0) { const uint32_t h = H[r1]; if (h == 0 || h >= k) return; }
    H[i] = k;
}

__device__ inline float box_area(const float* b)
{
    const float dx = b[1] - b[0], dy = b[3] - b[2], dz = b[5] - b[4];
    return dx * dy + dy * dz + dz * dx;
}

__device__ inline void kids2(const Node& q, int32_t* ref, float (*b)[6])
{
    ref[0] = __float_as_int(q.q3.x); ref[1] = __float_as_int(q.q3.y);
    b[0][0] = q.q0.x; b[0][1] = q.q0.y; b[0][2] = q.q0.z; b[0][3] = q.q0.w; b[0][4] = q.q1.x; b[0][5] = q.q1.y;
    b[1][0] = q.q1.z; b[1][1] = q.q1.w; b[1][2] = q.q2.x; b[1][3] = q.q2.y; b[1][4] = q.q2.z; b[1][5] = q.q2.w;
}

// one BVH4 node per work item: the BVH2 node's children, the inner child of largest area
// opened while fewer than four and while the stack budget allows one more push (the pushes
// above plus the children minus one, plus the tallest subtree below, within the budget)
__global__ __launch_bounds__(256) void k_c4_open(const C4Work* __restrict__ work, uint32_t nw, const Node* __restrict__ nodes,
                                                 const uint32_t* __restrict__ H, uint32_t budget, Node4* __restrict__ out4,
                                                 uint32_t* __restrict__ cnt, uint32_t* __restrict__ pnext, uint32_t* __restrict__ need)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nw) return;
    const C4Work w = work[i];
    int32_t ref[4];
    float b[4][6];
    kids2(nodes[w.i2], ref, b);
    int m = 2;
    while (m < 4) {
        int best = -1; float ba = -1.f;
        for (int k = 0; k < m; k++) if (ref[k] >= 0 && box_area(b[k]) > ba) { ba = box_area(b[k]); best = k; }
        if (best < 0) break;
        int32_t gr[2]; float gb[2][6];
        kids2(nodes[ref[best]], gr, gb);
        uint32_t hmax = 0;
        for (int k = 0; k < m; k++) if (k != best && ref[k] >= 0) hmax = max(hmax, H[ref[k]]);
        for (int j = 0; j < 2; j++) if (gr[j] >= 0) hmax = max(hmax, H[gr[j]]);
        if (w.P + (uint32_t)m + hmax > budget) break;
        ref[best] = gr[0]; for (int e = 0; e < 6; e++) b[best][e] = gb[0][e];
        ref[m] = gr[1]; for (int e = 0; e < 6; e++) b[m][e] = gb[1][e];
        m++;
    }
    const uint32_t P = w.P + (uint32_t)m - 1;
    atomicMax(need, P);
    Node4 nd;
    float* f = (float*)nd.q;
    int32_t* r = (int32_t*)&nd.q[6];
    uint32_t inner = 0;
    for (int k = 0; k < 4; k++) {
        for (int a = 0; a < 6; a++) f[4 * a + k] = k < m ? b[k][a] : 0.f;
        r[k] = k < m ? ref[k] : kNoChild;          // inner children: their BVH2 node until linked
        if (k < m && ref[k] >= 0) inner++;
    }
    nd.q[7] = make_float4(0.f, 0.f, 0.f, 0.f);
    out4[w.slot] = nd;
    cnt[i] = inner;
    pnext[i] = P;
}

// inner children get the next slots in work order (base + the item's prefix), and become
// the next level's work
__global__ __launch_bounds__(256) void k_c4_link(const C4Work* __restrict__ work, uint32_t nw, const uint32_t* __restrict__ prefix,
                                                 const uint32_t* __restrict__ pnext, uint32_t base, Node4* __restrict__ out4,
                                                 C4Work* __restrict__ next)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= nw) return;
    const C4Work w = work[i];
    int32_t* r = (int32_t*)&out4[w.slot].q[6];
    uint32_t j = prefix[i];
    for (int k = 0; k < 4; k++) {
        const int32_t c = r[k];
        if (c < 0 || c == kNoChild) continue;
        const uint32_t s = base + j;
        next[j] = C4Work{c, s, pnext[i]};
        r[k] = (int32_t)s;
        j++;
    }
}

// binary16 bits of the largest value <= x (DOWN) or the smallest >= x; beyond the range that is
// the largest finite value or infinity, whichever side is asked for
template <bool DOWN> __device__ inline uint16_t half_towards(double x)
{
    const float f = DOWN ? __double2float_rd(x) : __double2float_ru(x);
    const _Float16 h = (_Float16)f;
    uint16_t b;
    __builtin_memcpy(&b, &h, 2);
    if (DOWN ? (float)h <= f : (float)h >= f) return b;
    // one step of the ordered bits: away from zero when the value must grow in size
    if ((b & 0x7fffu) == 0u) return DOWN ? 0x8001u : 0x0001u;
    const bool neg = (b & 0x8000u) != 0u;
    return (uint16_t)(neg == DOWN ? b + 1u : b - 1u);
}

// Node4 -> NodeT: the origin is the middle of the node's box, so that the planes' distances
// from it are at most half its size (binary16 keeps 11 bits of them)
__global__ __launch_bounds__(256) void k_c4_pack(const Node4* __restrict__ in, uint32_t n, float scale, NodeT* __restrict__ out)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const Node4 nd = in[i];
    const float* f = (const float*)nd.q;
    const int32_t* ref = (const int32_t*)&nd.q[6];
    NodeT o;
    for (int k = 0; k < 4; k++) { o.ref[k] = ref[k]; o.pad0[k] = 0; o.pad1[k] = 0; }
    o.org[3] = 0.f;
    for (int a = 0; a < 3; a++) {
        const float* lo = f + 8 * a;
        const float* hi = lo + 4;
        float mn = 0.f, mx = 0.f;
        bool any = false;
        for (int k = 0; k < 4; k++)
            if (ref[k] != kNoChild) { mn = any ? fminf(mn, lo[k]) : lo[k]; mx = any ? fmaxf(mx, hi[k]) : hi[k]; any = true; }
        const float org = (0.5f * mn + 0.5f * mx) * scale;
        o.org[a] = org;
        uint16_t* q = a == 0 ? o.x : (a == 1 ? o.y : o.z);
        for (int k = 0; k < 4; k++) {
            const bool have = ref[k] != kNoChild;
            const uint16_t l = have ? half_towards<true>((double)lo[k] * (double)scale - (double)org) : (uint16_t)0;
            const uint16_t h = have ? half_towards<false>((double)hi[k] * (double)scale - (double)org) : (uint16_t)0;
            q[k] = l; q[4 + k] = h; q[8 + k] = l;
        }
    }
    out[i] = o;
}

inline void sfree(void* p) { if (p) (void)hipFree(p); }

} // namespace

int sah_rebuild_device(const int* d_first, const int* d_last, const int* d_split, int nprim, uint32_t leafmax, const Node* d_nodes,
                       Node** out_nodes, uint32_t* out_count, uint32_t* out_depth)
{
    *out_nodes = nullptr; *out_count = 0; *out_depth = 0;
    const int ni = nprim - 1;
    if (ni < 1) return 1;
    constexpr uint32_t kMaxLevels = 4096, kAhead = 4;    // levels launched between the host's looks
    uint32_t *flag, *pos, *tmp, *total, *dep;
    int* cb;
    SahLeaf *L0, *L1;
    SahTask *T0, *T1;
    SahBig* big;
    SahLevel* lev;
    Node* out = nullptr;
#define SK(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) { sfree(out); return hip_fail(e_, #x, __LINE__); } } while (0)
    const unsigned gb = (unsigned)((ni + 255) / 256);
    Scratch A, B;
    A.add(&flag, nprim); A.add(&pos, nprim); A.add(&tmp, scan_tmp_words((uint32_t)nprim)); A.add(&total, 1); A.add(&dep, 1); A.add(&cb, 6);
    A.add(&big, 1); A.add(&lev, kMaxLevels + kAhead + 2);
    if (int st = A.place()) return st;
    SK(hipMemsetAsync(flag, 0, 4 * (size_t)nprim, nullptr));
    SK(hipMemsetAsync(dep, 0, 4, nullptr));
    SK(hipMemsetAsync(lev, 0, sizeof(SahLevel) * (kMaxLevels + kAhead + 2), nullptr));
    k_sah_mark<<<gb, 256>>>(ni, d_first, d_last, d_split, leafmax, flag);
    SK(hipGetLastError());
    if (int st = scan_exclusive_u32(flag, pos, (uint32_t)nprim, total, tmp, nullptr)) return st;
    uint32_t n = 0;
    SK(hipMemcpy(&n, total, 4, hipMemcpyDeviceToHost));
    if (n < 2) return 1;
    const uint32_t cap = n / 2 + 1;
    B.add(&L0, n); B.add(&L1, n); B.add(&T0, cap); B.add(&T1, cap);
    if (int st = B.place()) return st;
    SK(hipMalloc(&out, sizeof(Node) * (size_t)(n - 1)));
    k_sah_gather<<<gb, 256>>>(ni, d_first, d_last, d_split, leafmax, d_nodes, pos, L0);
    // the root task: every leaf, its centroid bounds
    {
        const int init[6] = {0x7f7fffff, 0x7f7fffff, 0x7f7fffff, (int)0x80800000, (int)0x80800000, (int)0x80800000};
        SK(hipMemcpy(cb, init, 24, hipMemcpyHostToDevice));   // lo = max float, hi = ordered -max float
    }
    k_sah_root<<<std::min(1024u, (n + 255) / 256), 256>>>(L0, n, cb);
    k_sah_root_task<<<1, 64>>>(cb, n, T0, lev);
    SK(hipGetLastError());
    // While a level has tasks of kMidTask leaves or more, the host looks at every level: tasks of
    // at least kBigTask leaves go across the chip, and the host reads the task list while it
    // is short to find them.  Below that, kAhead levels are launched at a time, each taking its
    // number of tasks from the level before.  flag, pos and tmp are free by now and hold the
    // big tasks' flags, their prefix and the scan's scratch.
    constexpr uint32_t kHostTasks = 1024, kGrid = 16384, kNoLimit = 0xffffffffu;
    std::vector<SahTask> ht;
    std::vector<uint32_t> bigs;
    SahLevel now{1, n};
    SahLeaf *src = L0, *dst = L1;
    SahTask *tin = T0, *tout = T1;
    for (uint32_t level = 0; now.ntask;) {
        if (level > kMaxLevels) { sfree(out); return fail(LSG_ERR_INVALID, "sah_rebuild_device: no progress"); }
        if (now.maxm < kMidTask) {
            uint64_t bound = now.ntask;
            for (uint32_t j = 0; j < kAhead; j++, bound *= 2) {
                k_sah_level<64><<<(unsigned)std::min<uint64_t>(std::min<uint64_t>(bound, cap), kGrid), 64>>>(tin, lev + level, 0, kNoLimit, src, dst, out,
                                                                                                    tout, lev + level + 1, dep);
                level++;
                std::swap(src, dst);
                std::swap(tin, tout);
            }
        } else {
            bigs.clear();
            if (now.maxm >= kBigTask && now.ntask <= kHostTasks) {
                ht.resize(now.ntask);
                SK(hipMemcpy(ht.data(), tin, sizeof(SahTask) * now.ntask, hipMemcpyDeviceToHost));
                for (uint32_t i = 0; i < now.ntask; i++) if (ht[i].end - ht[i].begin >= kBigTask) bigs.push_back(i);
            }
            const unsigned grid = std::min(now.ntask, kGrid);
            k_sah_level<64><<<grid, 64>>>(tin, lev + level, 0, kMidTask, src, dst, out, tout, lev + level + 1, dep);
            k_sah_level<1024><<<std::min(grid, 1024u), 1024>>>(tin, lev + level, kMidTask, bigs.empty() ? kNoLimit : kBigTask, src, dst, out, tout,
                                                               lev + level + 1, dep);
            for (uint32_t i : bigs) {
                const SahTask* t = tin + i;
                const uint32_t m = ht[i].end - ht[i].begin;
                const unsigned g = std::min(2048u, (m + 255) / 256);
                k_big_init<<<1, 256>>>(big);
                k_big_bin<<<g, 256>>>(t, src, big);
                k_big_split<<<1, 64>>>(t, big);
                k_big_flag<<<g, 256>>>(t, src, big, flag);
                if (int st = scan_exclusive_u32(flag, pos, m, nullptr, tmp, nullptr)) { sfree(out); return st; }
                k_big_scatter<<<g, 256>>>(t, src, dst, flag, pos, big);
                k_big_emit<<<1, 64>>>(t, dst, big, out, tout, lev + level + 1, dep);
            }
            level++;
            std::swap(src, dst);
            std::swap(tin, tout);
        }
        SK(hipGetLastError());
        SK(hipMemcpy(&now, lev + level, sizeof now, hipMemcpyDeviceToHost));
        if (now.ntask > cap) { sfree(out); return fail(LSG_ERR_INVALID, "sah_rebuild_device: %u tasks over %u", now.ntask, cap); }
    }
    uint32_t d = 0;
    SK(hipMemcpy(&d, dep, 4, hipMemcpyDeviceToHost));
#undef SK
    *out_nodes = out; *out_count = n - 1; *out_depth = d;
    return 0;
}

// The BVH4 of a BVH2 (nodes, nn, root >= 0) on the GPU, breadth first: heights bottom-up
// (one launch per level),
// then one level of BVH4 nodes per launch, slots in level order.  budget = the traversal
// stack entries minus one.  Sets C.nnodes4, C.root4 = 0, C.stack_need.
int collapse4_device(ColliderImpl& C, uint32_t budget, Node4** nodes4)
{
    *nodes4 = nullptr;
    const uint32_t nn = C.nnodes;
    uint32_t *H, *cnt, *prefix, *pnext, *tmp, *total, *need;
    C4Work *w0, *w1;
    Node4* out = nullptr;
#define SK(x) do { hipError_t e_ = (x); if (e_ != hipSuccess) { sfree(out); return hip_fail(e_, #x, __LINE__); } } while (0)
    const unsigned gb = (nn + 255) / 256;
    Scratch A;
    A.add(&H, nn); A.add(&w0, nn); A.add(&w1, nn); A.add(&cnt, nn); A.add(&prefix, nn); A.add(&pnext, nn); A.add(&tmp, scan_tmp_words(nn));
    A.add(&total, 1); A.add(&need, 1);
    if (int st = A.place()) return st;
    SK(hipMemsetAsync(H, 0, 4 * (size_t)nn, nullptr));
    uint32_t hroot = 0;
    for (uint32_t k = 1;; k++) {
        k_c4_height<<<gb, 256>>>(nn, C.d_nodes, H, k);
        if (k % 8 == 0) {
            SK(hipMemcpy(&hroot, H + C.root, 4, hipMemcpyDeviceToHost));
            if (hroot) break;
            if (k > 4096) return fail(LSG_ERR_INVALID, "collapse4: no progress");
        }
    }
    SK(hipGetLastError());
    if (hroot > budget) return fail(LSG_ERR_LIMIT, "collapse4: tree height %u over stack budget %u", hroot, budget);
    SK(hipMalloc(&out, sizeof(Node4) * (size_t)nn));
    SK(hipMemset(need, 0, 4));
    {
        const C4Work r{C.root, 0u, 0u};
        SK(hipMemcpy(w0, &r, sizeof r, hipMemcpyHostToDevice));
    }
    uint32_t nw = 1, n4 = 1;
    while (nw) {
        if (n4 > nn) { sfree(out); return fail(LSG_ERR_INVALID, "collapse4: more BVH4 nodes than BVH2 nodes"); }
        const unsigned g = (nw + 255) / 256;
        k_c4_open<<<g, 256>>>(w0, nw, C.d_nodes, H, budget, out, cnt, pnext, need);
        if (int st = scan_exclusive_u32(cnt, prefix, nw, total, tmp, nullptr)) { sfree(out); return st; }
        k_c4_link<<<g, 256>>>(w0, nw, prefix, pnext, n4, out, w1);
        SK(hipGetLastError());
        uint32_t t = 0;
        SK(hipMemcpy(&t, total, 4, hipMemcpyDeviceToHost));
        n4 += t;
        nw = t;
        std::swap(w0, w1);
    }
    uint32_t sn = 0;
    SK(hipMemcpy(&sn, need, 4, hipMemcpyDeviceToHost));
#undef SK
    *nodes4 = out;
    C.nnodes4 = n4; C.root4 = 0; C.stack_need = sn;
    return LSG_OK;
}

int pack4_device(ColliderImpl& C, const Node4* nodes4)
{
    // the scene's size becomes 2^13 to 2^14: a plane's distance from its node's origin is far
    // from binary16's limit, and the boxes' inflation (1e-5 of the largest coordinate) far
    // above its smallest steps
    float ext = 0.f;
    for (int a = 0; a < 3; a++) ext = std::max(ext, C.bmax[a] - C.bmin[a]);
    int e = 0;
    if (ext > 0.f && std::isfinite(ext)) (void)std::frexp(ext, &e);
    C.scale = std::ldexp(1.f, std::min(100, std::max(-100, 14 - e)));
    const size_t n = C.nnodes4 ? C.nnodes4 : 1;
    LSG_HIP(hipMalloc(&C.d_nodes4, sizeof(NodeT) * n));
    C.bytes += sizeof(NodeT) * n;
    if (C.nnodes4) k_c4_pack<<<(C.nnodes4 + 255) / 256, 256>>>(nodes4, C.nnodes4, C.scale, C.d_nodes4);
    LSG_HIP(hipGetLastError());
    return LSG_OK;
}

} // namespace lsg
