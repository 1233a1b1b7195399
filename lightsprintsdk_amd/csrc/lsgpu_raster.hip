// lsgpu_raster.hip -- texel rasterisation of lightmaps on the GPU (gfx950).
//
// Produces what enumerateTexelsPartial (RRSolver/lightmap.cpp:83-404, steps 1-2) gives the
// final gather for an object: every texel the object's unwrap covers, the pieces
// (SubTexels, gather.h:60-65) of each triangle inside it, and the texel's coverage flags
// (gather.h:68-80) -- by a design of this library:
//   1. each triangle's candidate texels are the cells of its bounding box in texel units;
//   2. one lane per (triangle, candidate) clips the triangle against the texel's square
//      (four axis-aligned half-planes in texel-local coordinates), and counts the fan
//      pieces and coverage flags of the intersection polygon;
//   3. non-empty pairs are compacted in candidate order (triangle-major) and stable-sorted
//      by texel index, so a texel's pieces come in triangle order and texels row-major;
//   4. runs of one texel become texel records; every pair writes its pieces (corner
//      coordinates in triangle space, area) at its scanned offset.
// All objects of a bake go through these steps together: their texels' numbers do not overlap
// and grow with the object, so one sort gives every object's list in turn.  The steps are
// short (2 to 30 us a kernel for 20 maps of 256^2) and what an object costs is launches, waits and
// allocations; one object at a time, counted first and then rasterised again, a bake of 20
// objects with 50,000 triangles took 64 ms to set up, together 3.0.
// Kept from the reference because they are its interface: the flag bits, the 0.03-texel
// edge tolerance of the edge flags (lightmap.cpp:292), the quadrant rule for an edge that
// crosses both texel axes (lightmap.cpp:302-311), and areaInMapSpace = half the piece's
// area in uv units (the reference's triangle-space area times the triangle's map area).
#include "lsgpu_internal.h"
#include <algorithm>
#include <cmath>
#include <cstring>
#include <utility>
#include <vector>

namespace lsg {

namespace {

enum : uint32_t { QX0Y0 = 1, QX1Y0 = 2, QX0Y1 = 4, QX1Y1 = 8, EX0 = 16, EX1 = 32, EY0 = 64, EY1 = 128 };

// a triangle's uv corners, its candidate box of texels and its index in the mesh
struct TriBox { float2 u0, u1, u2; uint32_t x0, y0, w, id, obj; };

__global__ __launch_bounds__(256) void k_raster_boxes(const float* __restrict__ uv, const uint32_t* __restrict__ ids, uint32_t ntri,
                                                      const RasterObject* __restrict__ objs, uint32_t nobj,
                                                      TriBox* __restrict__ tb, uint32_t* __restrict__ cnt)
{
    const uint32_t t = blockIdx.x * 256 + threadIdx.x;
    if (t >= ntri) return;
    uint32_t lo = 0, hi = nobj;
    while (hi - lo > 1) { const uint32_t mid = (lo + hi) >> 1; if (objs[mid].tri_begin <= t) lo = mid; else hi = mid; }
    const uint32_t W = objs[lo].width, H = objs[lo].height;
    const float* u = uv + 6 * (size_t)t;
    const float fw = (float)W, fh = (float)H;
    const float2 p0 = make_float2(u[0] * fw, u[1] * fh), p1 = make_float2(u[2] * fw, u[3] * fh), p2 = make_float2(u[4] * fw, u[5] * fh);
    const float2 e1 = make_float2(p1.x - p0.x, p1.y - p0.y), e2 = make_float2(p2.x - p0.x, p2.y - p0.y);
    const float cr = e1.x * e2.y - e1.y * e2.x;
    TriBox b;
    b.u0 = make_float2(u[0], u[1]); b.u1 = make_float2(u[2], u[3]); b.u2 = make_float2(u[4], u[5]);
    b.id = ids[t];
    b.obj = lo;
    b.x0 = b.y0 = b.w = 0;
    uint32_t n = 0;
    const float lx = fminf(p0.x, fminf(p1.x, p2.x)), hx = fmaxf(p0.x, fmaxf(p1.x, p2.x));
    const float ly = fminf(p0.y, fminf(p1.y, p2.y)), hy = fmaxf(p0.y, fmaxf(p1.y, p2.y));
    if (cr != 0.f && isfinite(cr) && isfinite(lx) && isfinite(hx) && isfinite(ly) && isfinite(hy) && hx >= 0.f && hy >= 0.f &&
        lx < fw && ly < fh) {
        const uint32_t x0 = (uint32_t)floorf(fmaxf(lx, 0.f)), y0 = (uint32_t)floorf(fmaxf(ly, 0.f));
        const uint32_t x1 = min(W, (uint32_t)floorf(fminf(hx, fw)) + 1u), y1 = min(H, (uint32_t)floorf(fminf(hy, fh)) + 1u);
        if (x1 > x0 && y1 > y0) { b.x0 = x0; b.y0 = y0; b.w = x1 - x0; n = (x1 - x0) * (y1 - y0); }
    }
    tb[t] = b;
    cnt[t] = n;
}

// The triangle (q0, q1, q2, texel-local) clipped to the unit square by the half-planes
// x >= 0, x <= 1, y >= 0, y <= 1 in turn; vertices on a side count as inside, crossings are
// placed exactly on the side.  Consecutive repeats are dropped.  Returns the vertex count
// (0 when fewer than three distinct vertices or no area remain).
__device__ inline int texel_polygon(float2 q0, float2 q1, float2 q2, float2* out)
{
    float2 a[8], b[8];
    a[0] = q0; a[1] = q1; a[2] = q2;
    int n = 3;
#pragma unroll
    for (int side = 0; side < 4; side++) {
        const bool ax = side < 2;                  // clip on x or on y
        const float lim = (side & 1) ? 1.f : 0.f;
        const float sg = (side & 1) ? -1.f : 1.f;  // inside when sg * (c - lim) >= 0
        int m = 0;
        for (int i = 0; i < n; i++) {
            const float2 p = a[i == 0 ? n - 1 : i - 1], c = a[i];
            const float dp = sg * ((ax ? p.x : p.y) - lim), dc = sg * ((ax ? c.x : c.y) - lim);
            if ((dp >= 0.f) != (dc >= 0.f)) {
                const float s = dp / (dp - dc);
                float2 x = make_float2(p.x + (c.x - p.x) * s, p.y + (c.y - p.y) * s);
                if (ax) x.x = lim; else x.y = lim;
                b[m++] = x;
            }
            if (dc >= 0.f) b[m++] = c;
        }
        n = 0;
        for (int i = 0; i < m; i++)
            if (n == 0 || b[i].x != a[n - 1].x || b[i].y != a[n - 1].y) a[n++] = b[i];
        if (n > 1 && a[n - 1].x == a[0].x && a[n - 1].y == a[0].y) n--;
        if (n < 3) return 0;
    }
    float twice = 0.f;
    for (int i = 1; i + 1 < n; i++)
        twice += (a[i].x - a[0].x) * (a[i + 1].y - a[0].y) - (a[i].y - a[0].y) * (a[i + 1].x - a[0].x);
    if (twice == 0.f) return 0;
    for (int i = 0; i < n; i++) out[i] = a[i];
    return n;
}

// Coverage flags of a texel's polygon (texel-local, square [0,1]^2): edge bits for vertices
// within 0.03 texel of a side, quadrant bits for vertices strictly inside a quadrant around
// the centre, and for an edge that changes both the x and the y side of the centre, the two
// quadrants below or above (by the sign of its line's height at the centre's x) and the two
// left or right (by the sign of where it crosses the centre's height).
__device__ inline uint32_t coverage_flags(const float2* v, int n)
{
    constexpr float kErr = 0.03f;
    uint32_t f = 0;
    float px = v[n - 1].x - 0.5f, py = v[n - 1].y - 0.5f;
    for (int i = 0; i < n; i++) {
        const float x = v[i].x - 0.5f, y = v[i].y - 0.5f;
        f |= (x < -0.5f + kErr ? EX0 : 0u) | (x > 0.5f - kErr ? EX1 : 0u) | (y < -0.5f + kErr ? EY0 : 0u) | (y > 0.5f - kErr ? EY1 : 0u);
        if (x != 0.f && y != 0.f) f |= x < 0.f ? (y < 0.f ? QX0Y0 : QX0Y1) : (y < 0.f ? QX1Y0 : QX1Y1);
        if ((px < 0.f) != (x < 0.f) && (py < 0.f) != (y < 0.f)) {
            const float slope = (y - py) / (x - px);
            const float at0 = y - slope * x;              // the line's height at the centre's x
            f |= at0 < 0.f ? (QX0Y0 | QX1Y0) : (QX0Y1 | QX1Y1);
            f |= -at0 / slope < 0.f ? (QX0Y0 | QX0Y1) : (QX1Y0 | QX1Y1);
        }
        px = x; py = y;
    }
    return f;
}

// candidate c -> triangle (largest t with off[t] <= c), texel (x, y)
__device__ inline uint32_t candidate(const uint32_t* off, uint32_t ntri, const TriBox* tb, uint32_t c, uint32_t& x, uint32_t& y)
{
    uint32_t lo = 0, hi = ntri;
    while (hi - lo > 1) { const uint32_t mid = (lo + hi) >> 1; if (off[mid] <= c) lo = mid; else hi = mid; }
    const TriBox& b = tb[lo];
    const uint32_t k = c - off[lo];
    x = b.x0 + k % b.w;
    y = b.y0 + k / b.w;
    return lo;
}

// the triangle's corners relative to texel (x, y), each u * W - x with one rounding (a
// fused multiply-add), so they keep the precision of small local coordinates
__device__ inline float2 local_corner(float2 u, float fw, float fh, float ox, float oy)
{
    return make_float2(__fmaf_rn(u.x, fw, -ox), __fmaf_rn(u.y, fh, -oy));
}

__device__ inline int clip_candidate(const TriBox& b, uint32_t x, uint32_t y, float fw, float fh, float2* poly, float2& q0)
{
    const float ox = (float)x, oy = (float)y;
    q0 = local_corner(b.u0, fw, fh, ox, oy);
    return texel_polygon(q0, local_corner(b.u1, fw, fh, ox, oy), local_corner(b.u2, fw, fh, ox, oy), poly);
}

// per candidate: (pieces << 8 | flags), and 1 where the pair is not empty
__global__ __launch_bounds__(256) void k_raster_count(const uint32_t* __restrict__ off, uint32_t ntri, const TriBox* __restrict__ tb,
                                                      uint32_t C, const RasterObject* __restrict__ objs, uint16_t* __restrict__ info,
                                                      uint32_t* __restrict__ nz)
{
    const uint32_t c = blockIdx.x * 256 + threadIdx.x;
    if (c >= C) return;
    uint32_t x, y;
    const uint32_t t = candidate(off, ntri, tb, c, x, y);
    const RasterObject& o = objs[tb[t].obj];
    float2 poly[8], q0;
    const int n = clip_candidate(tb[t], x, y, (float)o.width, (float)o.height, poly, q0);
    info[c] = n ? (uint16_t)(((uint32_t)(n - 2) << 8) | coverage_flags(poly, n)) : (uint16_t)0;
    nz[c] = n ? 1u : 0u;
}

// keys: the texel's number from slot0 on
__global__ __launch_bounds__(256) void k_raster_compact(const uint32_t* __restrict__ off, uint32_t ntri, const TriBox* __restrict__ tb,
                                                        uint32_t C, const RasterObject* __restrict__ objs, uint32_t slot0,
                                                        const uint32_t* __restrict__ nz, const uint32_t* __restrict__ pos,
                                                        uint32_t* __restrict__ keys, uint32_t* __restrict__ vals)
{
    const uint32_t c = blockIdx.x * 256 + threadIdx.x;
    if (c >= C || !nz[c]) return;
    uint32_t x, y;
    const uint32_t t = candidate(off, ntri, tb, c, x, y);
    const RasterObject& o = objs[tb[t].obj];
    keys[pos[c]] = o.slot - slot0 + x + y * o.width;
    vals[pos[c]] = c;
}

// per sorted pair: its piece count, and 1 where a run of one texel starts
__global__ __launch_bounds__(256) void k_raster_runs(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ vals, uint32_t np,
                                                     const uint16_t* __restrict__ info, uint32_t* __restrict__ pieces,
                                                     uint32_t* __restrict__ head)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= np) return;
    pieces[i] = (uint32_t)info[vals[i]] >> 8;
    head[i] = (i == 0 || keys[i] != keys[i - 1]) ? 1u : 0u;
}

__global__ __launch_bounds__(256) void k_raster_texels(const uint32_t* __restrict__ keys, const uint32_t* __restrict__ vals, uint32_t np,
                                                       const uint16_t* __restrict__ info, const uint32_t* __restrict__ head,
                                                       const uint32_t* __restrict__ ord, const uint32_t* __restrict__ soff,
                                                       const RasterObject* __restrict__ objs, uint32_t nobj, uint32_t slot0,
                                                       uint32_t sub_base, lsg_texel* __restrict__ texels, uint32_t* __restrict__ too_many)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= np || !head[i]) return;
    const uint32_t key = keys[i];
    uint32_t count = 0, flags = 0;
    for (uint32_t j = i; j < np && keys[j] == key; j++) {
        const uint32_t q = info[vals[j]];
        count += q >> 8;
        flags |= q & 255u;
    }
    if (count > 0xffffu) { atomicMax(too_many, count); count = 0xffffu; }
    lsg_texel T;
    T.out_index = slot0 + key;
    T.sub_begin = sub_base + soff[i];
    T.sub_count_flags = count | (flags << 16);
    uint32_t lo = 0, hi = nobj;
    while (hi - lo > 1) { const uint32_t mid = (lo + hi) >> 1; if (objs[mid].slot - slot0 <= key) lo = mid; else hi = mid; }
    T.key = objs[lo].id * 0x9E3779B1u + (key - (objs[lo].slot - slot0));      // stable per-texel seed id
    texels[ord[i]] = T;
}

__global__ __launch_bounds__(256) void k_raster_emit(const uint32_t* __restrict__ off, uint32_t ntri, const TriBox* __restrict__ tb,
                                                     const uint32_t* __restrict__ vals, uint32_t np, const uint32_t* __restrict__ soff,
                                                     const RasterObject* __restrict__ objs, lsg_subtexel* __restrict__ subs)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= np) return;
    uint32_t x, y;
    const uint32_t t = candidate(off, ntri, tb, vals[i], x, y);
    const TriBox b = tb[t];
    const RasterObject& ob = objs[b.obj];
    const float fw = (float)ob.width, fh = (float)ob.height;
    const float area_scale = (float)(0.25 / ((double)ob.width * (double)ob.height));
    float2 poly[8], q0;
    const int n = clip_candidate(b, x, y, fw, fh, poly, q0);
    // triangle-space coordinates: p - corner 0 = a e1 + b e2, with the edges from the
    // texel-local corners
    const float2 q1 = local_corner(b.u1, fw, fh, (float)x, (float)y), q2 = local_corner(b.u2, fw, fh, (float)x, (float)y);
    const float2 e1 = make_float2(q1.x - q0.x, q1.y - q0.y), e2 = make_float2(q2.x - q0.x, q2.y - q0.y);
    const float inv = 1.f / (e1.x * e2.y - e1.y * e2.x);
    float2 tc[8];
    for (int k = 0; k < n; k++) {
        const float dx = poly[k].x - q0.x, dy = poly[k].y - q0.y;
        tc[k] = make_float2((dx * e2.y - dy * e2.x) * inv, (e1.x * dy - e1.y * dx) * inv);
    }
    lsg_subtexel* o = subs + soff[i];
    for (int k = 1; k + 1 < n; k++) {
        const float cr = (poly[k].x - poly[0].x) * (poly[k + 1].y - poly[0].y) - (poly[k].y - poly[0].y) * (poly[k + 1].x - poly[0].x);
        lsg_subtexel s;
        s.triangle = b.id;
        s.uv[0] = tc[0].x; s.uv[1] = tc[0].y;
        s.uv[2] = tc[k].x; s.uv[3] = tc[k].y;
        s.uv[4] = tc[k + 1].x; s.uv[5] = tc[k + 1].y;
        s.area = fabsf(cr) * area_scale;
        o[k - 1] = s;
    }
}

inline unsigned blocks(uint64_t n) { return (unsigned)((n + 255) / 256); }

constexpr uint64_t kGroupCandidates = 1ull << 26;        // candidates rasterised together, unless one object has more

// The texels and pieces of objects [o0, o1), whose triangles are [t0, t1) and have C
// candidates.  The counts are added to out; then, unless counts_only or out's caps are too
// small, the lists are appended to what out holds.
int raster_group(const RasterObject* objs, const RasterObject* d_objs, uint32_t o0, uint32_t o1, uint32_t t0, uint32_t t1, const TriBox* tb,
                 const uint32_t* cnt, uint32_t C, bool counts_only, RasterOut& out, hipStream_t st)
{
    if (!C) return LSG_OK;
    const uint32_t ntri = t1 - t0, slot0 = objs[o0].slot;
    int e;
    tb += t0;
    Scratch A;
    uint32_t *off, *tot, *nz, *pos, *tmp;
    uint16_t* info;
    A.add(&off, (size_t)ntri + 1); A.add(&tot, 4); A.add(&info, C); A.add(&nz, C); A.add(&pos, C);
    A.add(&tmp, std::max(scan_tmp_words(ntri), scan_tmp_words(C)));
    if ((e = A.place())) return e;
    if ((e = scan_exclusive_u32(cnt + t0, off, ntri, tot, tmp, st))) return e;
    k_raster_count<<<blocks(C), 256, 0, st>>>(off, ntri, tb, C, d_objs, info, nz);
    if ((e = scan_exclusive_u32(nz, pos, C, tot, tmp, st))) return e;
    uint32_t np = 0;
    LSG_HIP(hipMemcpyAsync(&np, tot, 4, hipMemcpyDeviceToHost, st));
    LSG_HIP(hipStreamSynchronize(st));
    if (!np) return LSG_OK;
    Scratch P;
    uint32_t *keys, *vals, *k2, *v2, *sorttmp, *pieces, *head, *soff, *ord, *ptmp;
    P.add(&keys, np); P.add(&vals, np); P.add(&k2, np); P.add(&v2, np); P.add(&sorttmp, sort_tmp_words(np)); P.add(&pieces, np);
    P.add(&head, np); P.add(&soff, np); P.add(&ord, np); P.add(&ptmp, scan_tmp_words(np));
    if ((e = P.place())) return e;
    k_raster_compact<<<blocks(C), 256, 0, st>>>(off, ntri, tb, C, d_objs, slot0, nz, pos, keys, vals);
    const uint64_t span = (uint64_t)objs[o1 - 1].slot - slot0 + (uint64_t)objs[o1 - 1].width * objs[o1 - 1].height;
    int bits = 1;
    while (bits < 32 && ((uint64_t)1 << bits) < span) bits++;
    if ((e = sort_pairs_u32(keys, vals, k2, v2, np, bits, sorttmp, st))) return e;
    k_raster_runs<<<blocks(np), 256, 0, st>>>(keys, vals, np, info, pieces, head);
    if ((e = scan_exclusive_u32(pieces, soff, np, tot, ptmp, st))) return e;
    if ((e = scan_exclusive_u32(head, ord, np, tot + 1, ptmp, st))) return e;
    uint32_t h[2] = {0, 0};
    LSG_HIP(hipMemcpyAsync(h, tot, 8, hipMemcpyDeviceToHost, st));
    LSG_HIP(hipStreamSynchronize(st));
    const uint32_t nt0 = out.ntex, ns0 = out.nsub;
    out.ntex += h[1]; out.nsub += h[0];
    if (counts_only || out.ntex > out.cap_t || out.nsub > out.cap_s) return LSG_OK;
    // room for the lists (grown by a copy when an earlier group has some)
    lsg_texel* T = nullptr;
    lsg_subtexel* S = nullptr;
    LSG_HIP(hipMalloc(&T, sizeof(lsg_texel) * (size_t)out.ntex));
    hipError_t he = hipMalloc(&S, sizeof(lsg_subtexel) * (size_t)out.nsub);
    if (he != hipSuccess) { (void)hipFree(T); return hip_fail(he, "hipMalloc", __LINE__); }
    std::swap(T, out.tex); std::swap(S, out.sub);
    if (nt0) he = hipMemcpyAsync(out.tex, T, sizeof(lsg_texel) * (size_t)nt0, hipMemcpyDeviceToDevice, st);
    if (he == hipSuccess && ns0) he = hipMemcpyAsync(out.sub, S, sizeof(lsg_subtexel) * (size_t)ns0, hipMemcpyDeviceToDevice, st);
    if (he == hipSuccess && (T || S)) he = hipStreamSynchronize(st);
    if (T) (void)hipFree(T);
    if (S) (void)hipFree(S);
    LSG_HIP(he);
    LSG_HIP(hipMemsetAsync(tot + 2, 0, 4, st));
    k_raster_texels<<<blocks(np), 256, 0, st>>>(keys, vals, np, info, head, ord, soff, d_objs + o0, o1 - o0, slot0, ns0, out.tex + nt0, tot + 2);
    k_raster_emit<<<blocks(np), 256, 0, st>>>(off, ntri, tb, vals, np, soff, d_objs, out.sub + ns0);
    LSG_HIP(hipGetLastError());
    uint32_t worst = 0;
    LSG_HIP(hipMemcpyAsync(&worst, tot + 2, 4, hipMemcpyDeviceToHost, st));
    LSG_HIP(hipStreamSynchronize(st));
    if (worst) return fail(LSG_ERR_LIMIT, "lsg_rasterize_texels: a texel has %u subtexels (at most 65535)", worst);
    return LSG_OK;
}

} // namespace

int raster_objects(const RasterObject* objs, uint32_t nobj, const float* const* uv, const uint32_t* const* ids, bool counts_only,
                   RasterOut& out, hipStream_t st)
{
    const uint64_t ntri64 = nobj ? (uint64_t)objs[nobj - 1].tri_begin + objs[nobj - 1].ntri : 0;
    if (!ntri64) return LSG_OK;
    const uint32_t ntri = (uint32_t)ntri64;
    int e;
    Scratch A;
    float* d_uv;
    uint32_t *d_ids, *cnt;
    TriBox* tb;
    RasterObject* d_objs;
    A.add(&d_uv, 6 * (size_t)ntri); A.add(&d_ids, ntri); A.add(&tb, ntri); A.add(&cnt, ntri); A.add(&d_objs, nobj);
    if ((e = A.place())) return e;
    std::vector<uint32_t> hc(7 * (size_t)ntri);          // uv and ids of all objects, later the candidate counts
    for (uint32_t o = 0; o < nobj; o++)
        if (objs[o].ntri) {
            memcpy(hc.data() + 6 * (size_t)objs[o].tri_begin, uv[o], 24 * (size_t)objs[o].ntri);
            memcpy(hc.data() + 6 * (size_t)ntri + objs[o].tri_begin, ids[o], 4 * (size_t)objs[o].ntri);
        }
    LSG_HIP(hipMemcpyAsync(d_uv, hc.data(), 24 * (size_t)ntri, hipMemcpyHostToDevice, st));
    LSG_HIP(hipMemcpyAsync(d_ids, hc.data() + 6 * (size_t)ntri, 4 * (size_t)ntri, hipMemcpyHostToDevice, st));
    LSG_HIP(hipMemcpyAsync(d_objs, objs, sizeof(RasterObject) * nobj, hipMemcpyHostToDevice, st));
    k_raster_boxes<<<blocks(ntri), 256, 0, st>>>(d_uv, d_ids, ntri, d_objs, nobj, tb, cnt);
    LSG_HIP(hipStreamSynchronize(st));                   // hc is read
    LSG_HIP(hipMemcpyAsync(hc.data(), cnt, 4 * (size_t)ntri, hipMemcpyDeviceToHost, st));
    LSG_HIP(hipStreamSynchronize(st));
    // 64-bit candidate sums (each box is at most W*H <= 2^28 cells), objects taken together up
    // to kGroupCandidates
    uint64_t sum = 0;
    for (uint32_t o = 0, o0 = 0; o < nobj; o++) {
        uint64_t c = 0;
        for (uint32_t t = objs[o].tri_begin; t < objs[o].tri_begin + objs[o].ntri; t++) c += hc[t];
        if (c >= (1ull << 31)) return fail(LSG_ERR_LIMIT, "lsg_rasterize_texels: %llu candidate texels", (unsigned long long)c);
        if (sum && sum + c > kGroupCandidates) {
            if ((e = raster_group(objs, d_objs, o0, o, objs[o0].tri_begin, objs[o].tri_begin, tb, cnt, (uint32_t)sum, counts_only, out, st))) return e;
            o0 = o; sum = 0;
        }
        sum += c;
        if (o + 1 == nobj) return raster_group(objs, d_objs, o0, nobj, objs[o0].tri_begin, ntri, tb, cnt, (uint32_t)sum, counts_only, out, st);
    }
    return LSG_OK;
}

} // namespace lsg

using namespace lsg;

extern "C" int lsg_rasterize_texels(const float* tri_uv, const uint32_t* tri_ids, uint32_t ntri, uint32_t width, uint32_t height,
                                    uint32_t object_id, lsg_texel* texels, uint32_t* ntexels, lsg_subtexel* subs, uint32_t* nsubs,
                                    uint32_t out_base)
{
    if (!ntexels || !nsubs || (ntri && (!tri_uv || !tri_ids))) return fail(LSG_ERR_INVALID, "lsg_rasterize_texels: null argument");
    if (!width || !height || (uint64_t)width * height > (1ull << 28))
        return fail(LSG_ERR_INVALID, "lsg_rasterize_texels: bad map size %ux%u", width, height);
    if (!device_ready()) return fail(LSG_ERR_NO_DEVICE, "lsg_rasterize_texels: no gfx950 device");
    const bool counts_only = !texels && !subs;
    if (!counts_only && (!texels || !subs)) return fail(LSG_ERR_INVALID, "lsg_rasterize_texels: give both output arrays");
    RasterOut out;
    out.cap_t = *ntexels; out.cap_s = *nsubs;
    const RasterObject ob{0, ntri, width, height, out_base, object_id};
    int r = raster_objects(&ob, 1, &tri_uv, &tri_ids, counts_only, out, nullptr);
    if (r) return r;
    *ntexels = out.ntex; *nsubs = out.nsub;
    if (counts_only) return LSG_OK;
    if (out.ntex > out.cap_t || out.nsub > out.cap_s)
        return fail(LSG_ERR_LIMIT, "lsg_rasterize_texels: need %u texels / %u subtexels", out.ntex, out.nsub);
    if (out.ntex) LSG_HIP(hipMemcpy(texels, out.tex, sizeof(lsg_texel) * (size_t)out.ntex, hipMemcpyDeviceToHost));
    if (out.nsub) LSG_HIP(hipMemcpy(subs, out.sub, sizeof(lsg_subtexel) * (size_t)out.nsub, hipMemcpyDeviceToHost));
    return LSG_OK;
}
