// lsgpu_internal.h -- shared host/device definitions of liblsgpu (gfx950).
//
// All float arithmetic that decides a hit is written in the reference's
// operation order and compiled with -ffp-contract=off and correctly rounded
// division/sqrt, so per-triangle accept/reject and hit distance are bit-identical
// to LightsprintCore's IT_BSP_FASTER triangle test (IntersectBspFast.cpp:189-252).
#pragma once
#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>
#include <string>
#include <utility>
#include <vector>
#include "lsgpu.h"

namespace lsg {

// ---- error plumbing ------------------------------------------------------------------
void set_error(const char* fmt, ...);
int fail(int code, const char* fmt, ...);
int hip_fail(hipError_t e, const char* what, int line);
bool device_ready();   // a gfx950 device is present and selected

#define LSG_HIP(call) do { hipError_t e_ = (call); if (e_ != hipSuccess) return ::lsg::hip_fail(e_, #call, __LINE__); } while (0)

// ---- tree layout ---------------------------------------------------------------------
// BVH2 node, 64 bytes, four float4 loads:
//   q0 = (lo0.x, hi0.x, lo0.y, hi0.y)   q1 = (lo0.z, hi0.z, lo1.x, hi1.x)
//   q2 = (lo1.y, hi1.y, lo1.z, hi1.z)   q3 = (ref0, ref1, 0, 0) as int bits
// ref >= 0: internal node index; ref < 0: leaf, start = (ref>>4)&0x7ffffff,
// count = (ref&15)+1 triangles in leaf order.
struct alignas(16) Node { float4 q0, q1, q2, q3; };

// BVH4 node, 128 bytes, collapsed from the BVH2 above (what tree files hold):
//   q[0] = lo.x of children 0..3   q[1] = hi.x   q[2] = lo.y   q[3] = hi.y
//   q[4] = lo.z                    q[5] = hi.z   q[6] = child refs (int bits)
// Refs as in the BVH2 (>= 0 inner BVH4 node, < 0 leaf); kNoChild marks an unused slot.
struct alignas(128) Node4 { float4 q[8]; };
constexpr int32_t kNoChild = 0x7ffffffe;

// The BVH4 node as every GPU traversal reads it, one cache line, five 16-byte loads.  The
// child planes are binary16 distances from the node's origin, in units of the tree's power-
// of-two scale, rounded outwards (lo down, hi up): the boxes only grow, so culling stays
// conservative, and v_fma_mix reads them at no cost.  Each axis holds lo[4] hi[4] lo[4]: a ray
// going up loads 16 bytes from the first lo (near, far planes), one going down from hi.
struct alignas(128) NodeT {
    uint16_t x[12], y[12];     // bytes 0 and 24
    int32_t ref[4];            // byte 48
    uint16_t z[12];            // byte 64
    uint16_t pad0[4];
    float org[4];              // byte 96: origin, scaled
    uint32_t pad1[4];
};
static_assert(sizeof(NodeT) == 128, "a node is one cache line");

// Triangle in leaf order, 48 bytes + 8 bytes meta (TriangleSRLNP,
// IntersectBspFast.h:33-49, with the projection-selected components pre-picked):
//   plane = n4;  sv = (s[x], s[y], s[z], intersectReal);  ev = (r[x], r[y], l[z], ir[z])
//   meta  = (original triangle index, intersectByte)
struct TriSoA { float4* plane; float4* sv; float4* ev; uint2* meta; };

constexpr uint32_t kLeafBit = 0x80000000u;
__host__ __device__ inline bool ref_is_leaf(int32_t r) { return r < 0; }
__host__ __device__ inline uint32_t leaf_start(int32_t r) { return ((uint32_t)r >> 4) & 0x7ffffffu; }
__host__ __device__ inline uint32_t leaf_count(int32_t r) { return ((uint32_t)r & 15u) + 1u; }
__host__ __device__ inline int32_t make_leaf(uint32_t start, uint32_t count) { return (int32_t)(kLeafBit | (start << 4) | (count - 1u)); }

// projection axes for intersectByte (IntersectBspFast.cpp:202-204): x,y from byte%3, z from byte/3
__host__ __device__ inline void srlnp_axes(int byte, int& x, int& y, int& z)
{
    int m = byte % 3, d = byte / 3;
    x = m; y = (m + 1) % 3; z = (d == 0) ? 2 : (d == 1 ? 0 : 1);
    if (byte > 8) { x = 2; y = 0; z = 1; }
}

__device__ inline float sel3(float a, float b, float c, int i) { return i == 0 ? a : (i == 1 ? b : c); }

// Box::intersect, RRCollider/geometry.cpp:38-86 (scalar path; minf/maxf are the
// reference's ternaries, not fminf, so NaN behaviour matches).
__host__ __device__ inline float rminf(float a, float b) { return a < b ? a : b; }
__host__ __device__ inline float rmaxf(float a, float b) { return a > b ? a : b; }
__device__ inline bool ref_box_intersect(const float3 mn, const float3 mx, const float3 o, const float3 d,
                                         float rmin, float rmax, float& lo, float& hi)
{
    float l1 = (mn.x - o.x) / d.x, l2 = (mx.x - o.x) / d.x;
    float lmin = rminf(l1, l2), lmax = rmaxf(l1, l2);
    l1 = (mn.y - o.y) / d.y; l2 = (mx.y - o.y) / d.y;
    lmin = rmaxf(rminf(l1, l2), lmin); lmax = rminf(rmaxf(l1, l2), lmax);
    l1 = (mn.z - o.z) / d.z; l2 = (mx.z - o.z) / d.z;
    lmin = rmaxf(rminf(l1, l2), lmin); lmax = rminf(rmaxf(l1, l2), lmax);
    lmin = rmaxf(rmin, lmin); lmax = rminf(rmax, lmax);
    lo = lmin; hi = lmax;
    return (lmax >= 0.f) & (lmax >= lmin);
}

// Plane distance (IntersectBspFast.cpp:349-352) of one triangle.
__device__ inline float plane_distance(const float4 n, const float3 o, const float3 d, float& ndotdir)
{
    ndotdir = d.x * n.x + d.y * n.y + d.z * n.z;
    float ndoto = o.x * n.x + o.y * n.y + o.z * n.z + n.w;
    return -ndoto / ndotdir;
}

// intersectByte's projection axes as a test reads them: bits 0-1 = x (y is the axis after
// it), bits 2-3 = z, bit 4 = degenerate (never hit), so a test selects components without
// the byte's division by 3
__host__ __device__ inline uint32_t srlnp_axes_code(int byte)
{
    int x, y, z;
    srlnp_axes(byte, x, y, z);
    return (uint32_t)x | (uint32_t)z << 2 | (byte > 8 ? 16u : 0u);
}

// intersect_triangleSRLNP (IntersectBspFast.cpp:189-252) at distance t already in range.
__device__ inline bool srlnp_hit(const float4 sv, const float4 ev, uint32_t axes, const float3 o, const float3 d, float t, float& u,
                                 float& v)
{
    const float px = o.x + d.x * t, py = o.y + d.y * t, pz = o.z + d.z * t;   // IntersectLinear.cpp:40-45
    const uint32_t x = axes & 3u, z = (axes >> 2) & 3u;
    const bool x0 = x == 0u, x1 = x == 1u;
    const float pX = x0 ? px : (x1 ? py : pz), pY = x0 ? py : (x1 ? pz : px);
    const float pZ = z == 0u ? px : (z == 1u ? py : pz);
    v = ((pY - sv.y) * ev.x - (pX - sv.x) * ev.y) * sv.w;
    u = (pZ - sv.z - ev.z * v) * ev.w;
    return !((v < 0) | (v > 1) | (u < 0) | (u + v > 1) | (axes >= 16u));
}

// ---- device-side collider view ---------------------------------------------------------
// The rest of a triangle's test record in leaf order, 48 bytes: projected edge data,
// (original index, intersectByte) and the byte's axes code, read together once a ray
// passes the plane test.
struct alignas(16) TriRest { float4 sv, ev; uint2 meta; uint32_t axes, pad; };

struct ColliderView {
    const Node* nodes;
    const NodeT* nodes4;
    float unscale;         // 1 / the nodes' scale
    int32_t root4;
    const float4* plane; const TriRest* rest;
    int32_t root;
    uint32_t nvalid;
    float3 bmin, bmax;     // inflated mesh box
};

struct ColliderImpl {
    uint32_t ntri = 0, nverts = 0, nvalid = 0, nnodes = 0, depth = 0, leaf = 4;
    uint32_t nnodes4 = 0, stack_need = 0;   // BVH4 nodes; worst-case traversal stack entries
    int32_t root4 = 0;
    NodeT* d_nodes4 = nullptr;
    float scale = 1.f;            // the nodes' power-of-two scale (pack4_device)
    int32_t root = 0;
    float bmin[3], bmax[3], margin = 0;
    float* d_verts = nullptr; uint32_t* d_idx = nullptr;
    Node* d_nodes = nullptr;
    float4* d_plane = nullptr; TriRest* d_rest = nullptr;
    uint32_t* d_slot = nullptr;   // leaf-order slot of each original triangle
    uint32_t flags = 0;           // lsg_build_params flags the tree was built with
    unsigned long long* d_queue = nullptr;   // ray-queue counters of closest-hit launches (a ring)
    mutable uint32_t queue_next = 0;   // next counter a launch takes (host atomic)
    uint64_t bytes = 0;
    double build_ms = 0;
    ColliderView view() const
    {
        ColliderView v;
        v.nodes = d_nodes; v.plane = d_plane; v.rest = d_rest;
        v.nodes4 = d_nodes4; v.root4 = root4; v.unscale = 1.f / scale;
        v.root = root; v.nvalid = nvalid;
        v.bmin = make_float3(bmin[0], bmin[1], bmin[2]);
        v.bmax = make_float3(bmax[0], bmax[1], bmax[2]);
        return v;
    }
};

int stack_size_for_depth(uint32_t depth);   // 0 when too deep
// the traversal kernels' stack (32 or 64 entries, 0 = too deep) for a built tree.  The
// 32-entry kernels address nodes and triangle records by 32-bit byte offsets, so a tree
// whose arrays pass 4 GB takes the 64-entry ones.
inline int traversal_stack(const ColliderImpl& C)
{
    const int st = stack_size_for_depth(C.depth);
    return st == 32 && (C.nnodes4 > (1u << 25) || C.nvalid > (1u << 26)) ? 64 : st;
}

// ---- device-wide primitives (lsgpu_prim.hip) --------------------------------------------
// words of scratch scan_exclusive_u32 needs for n values
size_t scan_tmp_words(uint32_t n);
// out[i] = in[0] + ... + in[i-1] (in != out); *total (device, optional) = the sum of all
int scan_exclusive_u32(const uint32_t* in, uint32_t* out, uint32_t n, uint32_t* total, uint32_t* tmp, hipStream_t st);
size_t sort_tmp_words(uint32_t n);
// stable sort of n (key, value) pairs by the low `bits` bits of the keys; the result is
// in keys/vals, keys_tmp/vals_tmp are n-word scratch
int sort_pairs_u32(uint32_t* keys, uint32_t* vals, uint32_t* keys_tmp, uint32_t* vals_tmp, uint32_t n, int bits,
                   uint32_t* tmp, hipStream_t st);
// SHA-1 of the concatenation a || b (lsgpu_hash.cpp)
void sha1(const void* a, size_t na, const void* b, size_t nb, uint8_t out[20]);
// RRHash::getFileName's cache file name for a hash (lsgpu_hash.cpp)
std::string cache_file_name(const uint8_t hash[20], uint32_t version, const char* location, const char* extension);
// The same rebuild on the GPU (lsgpu_sah.hip) from the LBVH's Karras arrays and nodes:
// *out_nodes (device, *out_count nodes, root 0) and its depth; 0 = rebuilt, 1 = fewer than
// two leaves, else an LSG_ERR_* code
int sah_rebuild_device(const int* d_first, const int* d_last, const int* d_split, int nprim, uint32_t leafmax, const Node* d_nodes,
                       Node** out_nodes, uint32_t* out_count, uint32_t* out_depth);
// The BVH4 of C's BVH2 on the GPU (lsgpu_sah.hip): C.nnodes4, root4, stack_need and the nodes
// (device, the caller's to free)
struct ColliderImpl;
int collapse4_device(ColliderImpl& C, uint32_t budget, Node4** nodes4);
// C.d_nodes4 and C.scale from the BVH4 nodes (device) of C's tree; C.bytes counts them
int pack4_device(ColliderImpl& C, const Node4* nodes4);
// SAH rebuild of a BVH2's inner nodes over its leaves (lsgpu_sah.cpp): 0 = rebuilt,
// 1 = fewer than two leaves, 2 = malformed tree
int sah_rebuild(const float* nodes, uint32_t nnodes, int32_t root, float* out, uint32_t* out_nodes, int32_t* out_root,
                uint32_t* out_depth);

// ---- scratch of the build steps ----------------------------------------------------------
// one allocation for a step's arrays: parts are added, then placed
struct Scratch {
    std::vector<std::pair<void**, size_t>> parts;
    void* base = nullptr;
    Scratch() = default;
    Scratch(const Scratch&) = delete;
    ~Scratch() { if (base) (void)hipFree(base); }
    template <class T> void add(T** p, size_t n) { parts.push_back({(void**)p, sizeof(T) * n}); }
    int place()
    {
        size_t n = 0;
        for (auto& q : parts) n += (q.second + 255) / 256 * 256;
        hipError_t e = hipMalloc(&base, n ? n : 256);
        if (e != hipSuccess) { base = nullptr; return hip_fail(e, "hipMalloc", __LINE__); }
        char* c = (char*)base;
        for (auto& q : parts) { *q.first = c; c += (q.second + 255) / 256 * 256; }
        return LSG_OK;
    }
};

// ---- texel rasterisation (lsgpu_raster.hip) ---------------------------------------------
struct RasterObject {
    uint32_t tri_begin, ntri;      // its triangles among all objects' (in object order)
    uint32_t width, height;
    uint32_t slot;                 // out_index of its texel (0, 0); objects' texels follow one another
    uint32_t id;
};
struct RasterOut {                 // device lists, texels of object after object
    lsg_texel* tex = nullptr;
    lsg_subtexel* sub = nullptr;
    uint32_t ntex = 0, nsub = 0;
    uint32_t cap_t = 0xffffffffu, cap_s = 0xffffffffu;     // with more than this, only the counts
    ~RasterOut() { if (tex) (void)hipFree(tex); if (sub) (void)hipFree(sub); }
};
// uv[o], ids[o]: host arrays of object o (6 floats and an index per triangle).  Synchronous on st.
int raster_objects(const RasterObject* objs, uint32_t nobj, const float* const* uv, const uint32_t* const* ids, bool counts_only,
                   RasterOut& out, hipStream_t st);

} // namespace lsg

struct lsg_collider { lsg::ColliderImpl impl; };
