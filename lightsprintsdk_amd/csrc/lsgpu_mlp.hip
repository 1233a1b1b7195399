// lsgpu_mlp.hip -- the learned-gather surrogate: a small MLP trained and run on gfx950
// matrix cores (v_mfma_f32_16x16x16_bf16: BF16 operands, FP32 accumulation).
//
// Network: 32 -> 64 -> 64 -> 64 -> 64 -> 4 (ReLU between layers), the last layer
// padded to 16 outputs so every GEMM dimension is a multiple of 16.  Inference and the
// training step are one kernel each, weights and activations in LDS; a training step adds a
// second one that sums the workgroups' gradients and takes the Adam step.  Activations are
// rounded to BF16 exactly where the products consume them; the CPU oracle rounds at the
// same points.
#include "lsgpu_internal.h"
#include <algorithm>
#include <vector>
#include <cstring>
#include <cmath>

typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v4f4 __attribute__((ext_vector_type(4), aligned(4)));      // a caller's floats

namespace lsg {

constexpr int kLayers = 5;
constexpr int kFeat = 32;                                  // input features per row
static const int kIn[kLayers] = {kFeat, 64, 64, 64, 64};
static const int kOut[kLayers] = {64, 64, 64, 64, 16};   // last layer: 4 used + 12 zero padding
constexpr int kOutUsed = 4;

__host__ __device__ inline uint16_t f2bf(float f)
{
    // round to nearest even (no NaN inputs here)
    uint32_t u;
    memcpy(&u, &f, 4);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (uint16_t)(u >> 16);
}
__host__ __device__ inline float bf2f(uint16_t b) { uint32_t u = (uint32_t)b << 16; float f; memcpy(&f, &u, 4); return f; }

// C[M x N] (fp32) = A[M x K] B[K x N] (bf16), all row-major: not on the network's path, but the same
// MFMA calls in the lane layout and the K order that k_mlp_infer and k_mlp_train build on, by
// themselves (lsg_mlp_gemm_test).  One wave per 16x16 tile, four waves per block.  Lane l feeds
// A row l%16 / B column l%16 with k = 4*(l/16)..+3 and receives C rows 4*(l/16)..+3 of column l%16.
__global__ __launch_bounds__(256) void k_gemm_bf16(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B, float* __restrict__ C,
                                                   int M, int N, int K)
{
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int tilesN = N / 16;
    const int tile = blockIdx.x * 4 + wave;
    if (tile >= (M / 16) * tilesN) return;
    const int tm = tile / tilesN, tn = tile % tilesN;
    const int r = lane & 15, kq = (lane >> 4) * 4;
    v4f acc = {0.f, 0.f, 0.f, 0.f};
    const uint16_t* Ar = A + (size_t)(tm * 16 + r) * K;
    const uint16_t* Bc = B + tn * 16 + r;
    for (int k0 = 0; k0 < K; k0 += 16) {
        v4s a, b;
        for (int i = 0; i < 4; i++) {
            a[i] = (short)Ar[k0 + kq + i];
            b[i] = (short)Bc[(size_t)(k0 + kq + i) * N];
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
    }
    for (int i = 0; i < 4; i++) C[(size_t)(tm * 16 + kq + i) * N + tn * 16 + r] = acc[i];
}

__global__ void k_to_bf16(const float* __restrict__ x, uint16_t* __restrict__ y, uint32_t n)
{
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) y[i] = f2bf(x[i]);
}

// Inference in one launch: the whole network per 16-row tile, one tile per wave at a
// time, four waves per workgroup, workgroups striding over 64-row groups (the weights are
// loaded into LDS once per workgroup).  The weights (transposed, BF16) and biases sit in LDS; each
// wave's activations ping-pong between two LDS tiles.  The products are the same MFMA
// calls in the same order as k_gemm_bf16's (same lane layout, same K steps); bias, ReLU and
// BF16 rounding come at the points the training step has them.
// LDS rows are padded by 4 elements (8 bytes): 16 lanes reading 16 rows at one column
// then hit 16 different bank pairs instead of one bank (row pitches of 64/128 bytes)
constexpr int kPad = 4;
constexpr int kWElems = (kFeat + kPad) * 64 + 3 * (64 + kPad) * 64 + (64 + kPad) * 16;
constexpr int kBElems = 4 * 64 + 16;
constexpr uint32_t kInferBlocks = 2048;                   // workgroups of the grid-stride inference launch
struct MlpOffsets { uint32_t w[kLayers]; uint32_t b[kLayers]; };

__global__ __launch_bounds__(256) void k_mlp_infer(const float* __restrict__ x, uint32_t n, const uint16_t* __restrict__ wb,
                                                   const float* __restrict__ p, MlpOffsets off, float* __restrict__ y)
{
    constexpr int kInL[kLayers] = {kFeat, 64, 64, 64, 64};
    constexpr int kOutL[kLayers] = {64, 64, 64, 64, 16};
    __shared__ __attribute__((aligned(16))) uint16_t wt[kWElems];   // layer l at tofs: W_l transposed, [out][in]
    __shared__ float bias[kBElems];
    __shared__ __attribute__((aligned(16))) uint16_t act[4][2][16 * (64 + kPad)];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    int tofs = 0, bofs = 0;
    for (int l = 0; l < kLayers; l++) {
        const int in = kInL[l], out = kOutL[l];
        for (int e = tid; e < in * out; e += 256) {
            const int k = e / out, c = e % out;
            wt[tofs + c * (in + kPad) + k] = wb[off.w[l] + e];
        }
        for (int c = tid; c < out; c += 256) bias[bofs + c] = p[off.b[l] + c];
        tofs += (in + kPad) * out; bofs += out;
    }
    __syncthreads();                                 // weights and biases in place
    const int r = lane & 15, kq = (lane >> 4) * 4;
    // each wave owns its activation tiles: within the tile loop only the wave's own LDS
    // writes must be visible to its lanes (no workgroup barrier)
    auto wave_sync = []() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    // grid-stride over 64-row groups: the weights are loaded into LDS once per workgroup
    const uint32_t groups = (uint32_t)(((uint64_t)n + 63) / 64);
    for (uint32_t it = blockIdx.x; it < groups; it += gridDim.x) {
    const uint64_t row0 = ((uint64_t)it * 4u + (uint32_t)wave) * 16u;
    uint16_t* A = act[wave][0];
    uint16_t* B = act[wave][1];
    for (int e = lane; e < 16 * kFeat; e += 64) {
        const uint32_t rr = (uint32_t)(e / kFeat), k = (uint32_t)(e % kFeat);
        A[rr * (kFeat + kPad) + k] = f2bf(row0 + rr < n ? x[(size_t)(row0 + rr) * kFeat + k] : 0.f);
    }
    wave_sync();
    tofs = 0; bofs = 0;
    for (int l = 0; l < kLayers; l++) {
        const int in = kInL[l], out = kOutL[l];
        const uint16_t* W = wt + tofs;
        for (int tile = 0; tile < out / 16; tile++) {
            v4f acc = {0.f, 0.f, 0.f, 0.f};
            for (int k0 = 0; k0 < in; k0 += 16) {
                // four consecutive BF16 values per operand: one 8-byte LDS read each
                // (offsets are multiples of 4 elements: pitches, k0 and kq are)
                const v4s a = *(const v4s*)(A + r * (in + kPad) + k0 + kq);
                const v4s b = *(const v4s*)(W + (tile * 16 + r) * (in + kPad) + k0 + kq);
                acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
            }
            const int col = tile * 16 + r;
            const float bb = bias[bofs + col];
            for (int i = 0; i < 4; i++) {
                const float z = acc[i] + bb;
                if (l < kLayers - 1) B[(kq + i) * (out + kPad) + col] = f2bf(z > 0.f ? z : 0.f);
                else if (col < kOutUsed && row0 + kq + i < n) y[(size_t)(row0 + kq + i) * kOutUsed + col] = z;
            }
        }
        wave_sync();
        uint16_t* t = A; A = B; B = t;
        tofs += (in + kPad) * out; bofs += out;
    }
    }
}

// One training step's gradients: forward, loss and backward of 64 rows at a time per
// workgroup (16 per wave), everything in LDS, the weight gradients of all its rows in MFMA
// accumulators (15 tiles per wave), then one partial sum per workgroup in memory.
//   forward   Z^T = W^T A^T: a lane gets four consecutive outputs of one row, so activations
//             are written as 8-byte pieces of rows, which the next product's operand reads
//   backward  dA^T = W dZ^T in the same form, masked by the layer's activations
//   dW        = A^T dZ over the workgroup's 64 rows: both operands are read along the rows
//             of transposed copies (feature-major) written beside the row-major ones
// Biases' gradients sum the unrounded dZ.  Loss of row i: sum_c (y_ic - t_ic)^2 + lambda (y_i3 -
// e_i)^2, e_i = sqrt(mean_c (y_ic - t_ic)^2) held constant, averaged over the n rows.
//
// Bound by the chain of ten small products and their barriers, 30 us a workgroup; the products
// are 0.9 GFLOP a step of 8192 rows, 1 us of the matrix cores.  Before, a launch per product and
// elementwise pass (26 a step), with dW by 16 to 64 waves that each walked all rows: 0.98 ms a
// step of 8192 rows -> 37 us (30 us + 5 us of k_mlp_update).
constexpr int kRows = 64, kPitch = kRows + kPad;         // rows per workgroup pass; LDS pitch of 64-wide rows
constexpr uint32_t kTrainBlocks = 256;                   // workgroups of a step, at most (one per CU)
constexpr int kWtElems = 64 * (kFeat + kPad) + 3 * 64 * (64 + kPad) + 16 * (64 + kPad);
constexpr int kWrElems = 3 * 64 * (64 + kPad) + 64 * (16 + kPad);

__device__ inline void put4(uint16_t* p, v4f v)
{
    v4s b;
    for (int i = 0; i < 4; i++) b[i] = (short)f2bf(v[i]);
    *(v4s*)p = b;
}

__global__ __launch_bounds__(256) void k_mlp_train(const float* __restrict__ x, const float* __restrict__ t, uint32_t n, float lambda,
                                                   const uint16_t* __restrict__ wb, const float* __restrict__ p, MlpOffsets off,
                                                   uint32_t nparams, float* __restrict__ partial, float* __restrict__ loss_part)
{
    __shared__ __attribute__((aligned(16))) uint16_t wt[kWtElems];           // W_l transposed, [out][in]
    __shared__ __attribute__((aligned(16))) uint16_t wr[kWrElems];           // W_l of layers 1..4, [in][out]
    __shared__ __attribute__((aligned(16))) uint16_t actT[(kFeat + 4 * 64) * kPitch];   // inputs of layer l, [feature][row]
    __shared__ __attribute__((aligned(16))) uint16_t dzT[2][64 * kPitch];    // dZ of a layer, [output][row]
    __shared__ __attribute__((aligned(16))) uint16_t rowbuf[4][2][16 * (64 + kPad)];    // a wave's rows, [row][feature]
    __shared__ float bias[kBElems], dbsum[4][kBElems], lsum[4];
    constexpr int kInL[kLayers] = {kFeat, 64, 64, 64, 64}, kOutL[kLayers] = {64, 64, 64, 64, 16};
    constexpr int kTofs[kLayers] = {0, 64 * (kFeat + kPad), 64 * (kFeat + kPad) + 64 * (64 + kPad), 64 * (kFeat + kPad) + 2 * 64 * (64 + kPad),
                                    64 * (kFeat + kPad) + 3 * 64 * (64 + kPad)};
    constexpr int kRofs[kLayers] = {0, 0, 64 * (64 + kPad), 2 * 64 * (64 + kPad), 3 * 64 * (64 + kPad)};
    constexpr int kAofs[kLayers] = {0, kFeat * kPitch, (kFeat + 64) * kPitch, (kFeat + 128) * kPitch, (kFeat + 192) * kPitch};
    constexpr int kBofs[kLayers] = {0, 64, 128, 192, 256};
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r = lane & 15, kq = (lane >> 4) * 4;
#pragma unroll
    for (int l = 0; l < kLayers; l++) {
        const int in = kInL[l], out = kOutL[l];
        for (int e = tid * 4; e < in * out; e += 1024) {
            const int k = e / out, c = e % out;
            const v4s w = *(const v4s*)(wb + off.w[l] + e);
            for (int i = 0; i < 4; i++) wt[kTofs[l] + (c + i) * (in + kPad) + k] = (uint16_t)w[i];
            if (l) *(v4s*)(wr + kRofs[l] + k * (out + kPad) + c) = w;
        }
        for (int c = tid; c < out; c += 256) bias[kBofs[l] + c] = p[off.b[l] + c];
    }
    auto wave_sync = []() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    const v4f zero = {0.f, 0.f, 0.f, 0.f};
    v4f dw0[2], dw1[4], dw2[4], dw3[4], dw4 = zero, db[4][4], db4 = zero;
#pragma unroll
    for (int i = 0; i < 4; i++) { dw1[i] = zero; dw2[i] = zero; dw3[i] = zero; for (int l = 0; l < 4; l++) db[l][i] = zero; }
    dw0[0] = zero; dw0[1] = zero;
    float loss = 0.f;
    const int myrow = wave * 16 + r;                     // the lane's row (column of the transposed products) in the pass
    const uint64_t passes = ((uint64_t)n + kRows - 1) / kRows;
    for (uint64_t ps = blockIdx.x; ps < passes; ps += gridDim.x) {
        __syncthreads();                                 // weights in place; the previous pass is read
        uint16_t* cur = rowbuf[wave][0];
        uint16_t* nxt = rowbuf[wave][1];
        {
            // rows of x, four lanes each; rows past the batch are zero
            const int rr = lane >> 2, k0 = (lane & 3) * 8;
            const uint64_t row = ps * kRows + (uint64_t)(wave * 16 + rr);
            v4f a = zero, b = zero;
            if (row < n) { a = *(const v4f4*)(x + row * kFeat + k0); b = *(const v4f4*)(x + row * kFeat + k0 + 4); }
            put4(cur + rr * (kFeat + kPad) + k0, a);
            put4(cur + rr * (kFeat + kPad) + k0 + 4, b);
            for (int i = 0; i < 4; i++) {
                actT[(k0 + i) * kPitch + wave * 16 + rr] = f2bf(a[i]);
                actT[(k0 + 4 + i) * kPitch + wave * 16 + rr] = f2bf(b[i]);
            }
        }
        wave_sync();
        const uint64_t row = ps * kRows + (uint64_t)myrow;
        v4f y = zero;
        uint32_t on[kLayers - 1] = {};                   // outputs past the ReLU, 16 bits a layer
#pragma unroll
        for (int l = 0; l < kLayers; l++) {
            const int in = kInL[l], out = kOutL[l];
#pragma unroll
            for (int mt = 0; mt < out / 16; mt++) {
                v4f acc = zero;
#pragma unroll
                for (int k0 = 0; k0 < in; k0 += 16)
                    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(*(const v4s*)(wt + kTofs[l] + (mt * 16 + r) * (in + kPad) + k0 + kq),
                                                                    *(const v4s*)(cur + r * (in + kPad) + k0 + kq), acc, 0, 0, 0);
                const int o = mt * 16 + kq;
                for (int i = 0; i < 4; i++) acc[i] += bias[kBofs[l] + o + i];
                if (l < kLayers - 1) {
                    for (int i = 0; i < 4; i++) {
                        if (acc[i] > 0.f) on[l] |= 1u << (mt * 4 + i);
                        else acc[i] = 0.f;
                    }
                    put4(nxt + r * (64 + kPad) + o, acc);
                    for (int i = 0; i < 4; i++) actT[kAofs[l < kLayers - 1 ? l + 1 : 0] + (o + i) * kPitch + myrow] = f2bf(acc[i]);
                } else y = acc;
            }
            wave_sync();
            uint16_t* s = cur; cur = nxt; nxt = s;
        }
        // loss and dY: the lanes with kq = 0 hold a row's four outputs
        v4f g = zero;
        if (kq == 0 && row < n) {
            const float* ti = t + row * 3;
            float se = 0.f;
            for (int c = 0; c < 3; c++) { const float d = y[c] - ti[c]; se += d * d; g[c] = 2.f * d / (float)n; }
            const float e = sqrtf(se / 3.f), de = y[3] - e;
            g[3] = 2.f * lambda * de / (float)n;
            loss += se + lambda * de * de;
        }
        put4(nxt + r * (16 + kPad) + kq, g);
        for (int i = 0; i < 4; i++) { dzT[0][(kq + i) * kPitch + myrow] = f2bf(g[i]); db4[i] += g[i]; }
        __syncthreads();
        // dW of a layer: this wave's tiles, over the pass's 64 rows
        auto grad = [&](const uint16_t* A, const uint16_t* D, int mi, int ni, v4f acc) {
#pragma unroll
            for (int k0 = 0; k0 < kRows; k0 += 16)
                acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(*(const v4s*)(A + (mi * 16 + r) * kPitch + k0 + kq),
                                                                *(const v4s*)(D + (ni * 16 + r) * kPitch + k0 + kq), acc, 0, 0, 0);
            return acc;
        };
#pragma unroll
        for (int l = kLayers - 1; l >= 0; l--) {
            const uint16_t* A = actT + kAofs[l];
            const uint16_t* D = dzT[(kLayers - 1 - l) & 1];
            if (l == 4) dw4 = grad(A, D, wave, 0, dw4);
            else if (l == 0) { for (int i = 0; i < 2; i++) dw0[i] = grad(A, D, i, wave, dw0[i]); }
            else {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (l == 3) dw3[i] = grad(A, D, i, wave, dw3[i]);
                    else if (l == 2) dw2[i] = grad(A, D, i, wave, dw2[i]);
                    else dw1[i] = grad(A, D, i, wave, dw1[i]);
                }
            }
            if (l == 0) break;
            // dA through the layer, masked by where its input passed the ReLU: the layer below's dZ
            uint16_t* s = cur; cur = nxt; nxt = s;       // cur = this layer's dZ rows
            wave_sync();
            const int out = kOutL[l];
            uint16_t* E = dzT[(kLayers - l) & 1];
#pragma unroll
            for (int mt = 0; mt < 4; mt++) {
                v4f acc = zero;
#pragma unroll
                for (int k0 = 0; k0 < out; k0 += 16)
                    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(*(const v4s*)(wr + kRofs[l] + (mt * 16 + r) * (out + kPad) + k0 + kq),
                                                                    *(const v4s*)(cur + r * (out + kPad) + k0 + kq), acc, 0, 0, 0);
                const int o = mt * 16 + kq;
                for (int i = 0; i < 4; i++) acc[i] = on[l - 1] >> (mt * 4 + i) & 1u ? acc[i] : 0.f;
                db[l - 1][mt] += acc;
                put4(nxt + r * (64 + kPad) + o, acc);
                for (int i = 0; i < 4; i++) E[(o + i) * kPitch + myrow] = f2bf(acc[i]);
            }
            __syncthreads();
        }
    }
    // this workgroup's partial sums
    float* P = partial + (size_t)blockIdx.x * nparams;
    auto store = [&](int l, int mi, int ni, v4f a) {
        for (int i = 0; i < 4; i++) P[off.w[l] + (mi * 16 + kq + i) * kOutL[l] + ni * 16 + r] = a[i];
    };
    store(4, wave, 0, dw4);
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if (i < 2) store(0, i, wave, dw0[i]);
        store(1, i, wave, dw1[i]); store(2, i, wave, dw2[i]); store(3, i, wave, dw3[i]);
    }
    // biases: over the lanes of one output, then over the waves
    auto over_rows = [&](float v) { for (int o = 8; o; o >>= 1) v += __shfl_xor(v, o); return v; };
#pragma unroll
    for (int i = 0; i < 4; i++) {
#pragma unroll
        for (int l = 0; l < 4; l++)
#pragma unroll
            for (int mt = 0; mt < 4; mt++) {
                const float v = over_rows(db[l][mt][i]);
                if (r == 0) dbsum[wave][kBofs[l] + mt * 16 + kq + i] = v;
            }
        const float v = over_rows(db4[i]);
        if (r == 0) dbsum[wave][kBofs[4] + kq + i] = v;
    }
    loss = over_rows(loss);
    if (lane == 0) lsum[wave] = loss;
    __syncthreads();
#pragma unroll
    for (int l = 0; l < kLayers; l++)
        for (int c = tid; c < kOutL[l]; c += 256) {
            const int b = kBofs[l] + c;
            P[off.b[l] + c] = (dbsum[0][b] + dbsum[1][b]) + (dbsum[2][b] + dbsum[3][b]);
        }
    if (tid == 0) loss_part[blockIdx.x] = (lsum[0] + lsum[1]) + (lsum[2] + lsum[3]);
}

// the workgroups' partial gradients added (64 parameters per workgroup, four lanes' shares of
// the parts each, in a fixed order) and, with lr > 0, the Adam step (Kingma & Ba 2015) on
// the fp32 master parameters and their BF16 copies; mask keeps the padded outputs.  The first
// workgroup also adds the loss.
struct AdamArgs { float* p; float* m; float* v; uint16_t* wb; const uint8_t* mask; float lr, b1, b2, eps, c1, c2; };

__global__ __launch_bounds__(256) void k_mlp_update(const float* __restrict__ partial, uint32_t parts, uint32_t nparams, float* __restrict__ g,
                                                    AdamArgs A, const float* __restrict__ loss_part, float* __restrict__ loss)
{
    __shared__ float s[4][64];
    const uint32_t c = threadIdx.x & 63u, q = threadIdx.x >> 6, i = blockIdx.x * 64 + c;
    float sum = 0.f;
    if (i < nparams) {
#pragma unroll 8
        for (uint32_t w = q; w < parts; w += 4) sum += partial[(size_t)w * nparams + i];
    }
    s[q][c] = sum;
    __syncthreads();
    if (q == 0 && i < nparams) {
        const float gi = (s[0][c] + s[1][c]) + (s[2][c] + s[3][c]);
        g[i] = gi;
        if (A.lr > 0 && A.mask[i]) {
            const float mi = A.b1 * A.m[i] + (1.f - A.b1) * gi;
            const float vi = A.b2 * A.v[i] + (1.f - A.b2) * gi * gi;
            A.m[i] = mi; A.v[i] = vi;
            const float pi = A.p[i] - A.lr * (mi / A.c1) / (sqrtf(vi / A.c2) + A.eps);
            A.p[i] = pi;
            A.wb[i] = f2bf(pi);
        }
    }
    if (blockIdx.x == 0) {
        __syncthreads();
        s[q][c] = threadIdx.x < parts ? loss_part[threadIdx.x] : 0.f;
        __syncthreads();
        float* f = &s[0][0];
        for (uint32_t w = 128; w; w >>= 1) {
            if (threadIdx.x < w) f[threadIdx.x] += f[threadIdx.x + w];
            __syncthreads();
        }
        if (threadIdx.x == 0) *loss = f[0];
    }
}
static_assert(kTrainBlocks <= 256, "k_mlp_update adds at most 256 losses");

static inline unsigned nb(uint64_t n) { return (unsigned)((n + 255) / 256); }

struct MlpImpl {
    uint32_t max_batch = 0;
    size_t wofs[kLayers], bofs[kLayers], nparams = 0;
    float* d_p = nullptr; float* d_g = nullptr; float* d_m = nullptr; float* d_v = nullptr; uint8_t* d_mask = nullptr;
    uint16_t* d_wb = nullptr;                    // bf16 weights (same offsets as d_p; biases unused)
    float* d_part = nullptr;                     // partial gradients of a step's workgroups, then their losses
    float* d_loss = nullptr;
    uint64_t step = 0;
    ~MlpImpl()
    {
        auto f = [](void* p) { if (p) (void)hipFree(p); };
        f(d_p); f(d_g); f(d_m); f(d_v); f(d_mask); f(d_wb); f(d_part); f(d_loss);
    }
};

} // namespace lsg

struct lsg_mlp { lsg::MlpImpl impl; };

using namespace lsg;

extern "C" {

int lsg_mlp_create(uint32_t max_batch, lsg_mlp** out)
{
    if (!out) return fail(LSG_ERR_INVALID, "lsg_mlp_create: out is null");
    *out = nullptr;
    if (!max_batch || max_batch % 16 || max_batch > (1u << 22)) return fail(LSG_ERR_INVALID, "max_batch must be a positive multiple of 16, <= 4M");
    if (!device_ready()) return fail(LSG_ERR_NO_DEVICE, "lsg_mlp_create: no gfx950 device");
    lsg_mlp* m = new (std::nothrow) lsg_mlp;
    if (!m) return fail(LSG_ERR_OOM, "host allocation");
    MlpImpl& M = m->impl;
    M.max_batch = max_batch;
    size_t o = 0;
    for (int l = 0; l < kLayers; l++) { M.wofs[l] = o; o += (size_t)kIn[l] * kOut[l]; M.bofs[l] = o; o += kOut[l]; }
    M.nparams = o;
    hipError_t e;
#define AL(p, bytes) do { if ((e = hipMalloc(&(p), (bytes))) != hipSuccess) { delete m; return hip_fail(e, "hipMalloc", __LINE__); } } while (0)
    AL(M.d_p, 4 * o); AL(M.d_g, 4 * o); AL(M.d_m, 4 * o); AL(M.d_v, 4 * o); AL(M.d_mask, o); AL(M.d_wb, 2 * o);
    AL(M.d_part, 4 * ((size_t)kTrainBlocks * o + kTrainBlocks));
    AL(M.d_loss, 16);
#undef AL
    std::vector<uint8_t> mask(o, 1);
    for (size_t r = 0; r < (size_t)kIn[kLayers - 1]; r++)
        for (int c = kOutUsed; c < kOut[kLayers - 1]; c++) mask[M.wofs[kLayers - 1] + r * kOut[kLayers - 1] + c] = 0;
    for (int c = kOutUsed; c < kOut[kLayers - 1]; c++) mask[M.bofs[kLayers - 1] + c] = 0;
    if ((e = hipMemcpy(M.d_mask, mask.data(), o, hipMemcpyHostToDevice)) != hipSuccess) { delete m; return hip_fail(e, "h2d", __LINE__); }
    (void)hipMemset(M.d_p, 0, 4 * o); (void)hipMemset(M.d_m, 0, 4 * o); (void)hipMemset(M.d_v, 0, 4 * o);
    *out = m;
    return LSG_OK;
}

void lsg_mlp_destroy(lsg_mlp* m) { delete m; }

uint32_t lsg_mlp_num_params(void)
{
    uint32_t o = 0;
    for (int l = 0; l < kLayers; l++) o += (uint32_t)(kIn[l] * kOut[l] + kOut[l]);
    return o;
}

int lsg_mlp_set_params(lsg_mlp* m, const float* params)
{
    if (!m || !params) return fail(LSG_ERR_INVALID, "lsg_mlp_set_params: null argument");
    MlpImpl& M = m->impl;
    std::vector<float> p(params, params + M.nparams);
    // padded outputs of the last layer stay exactly zero
    for (size_t r = 0; r < (size_t)kIn[kLayers - 1]; r++)
        for (int c = kOutUsed; c < kOut[kLayers - 1]; c++) p[M.wofs[kLayers - 1] + r * kOut[kLayers - 1] + c] = 0.f;
    for (int c = kOutUsed; c < kOut[kLayers - 1]; c++) p[M.bofs[kLayers - 1] + c] = 0.f;
    LSG_HIP(hipMemcpy(M.d_p, p.data(), 4 * M.nparams, hipMemcpyHostToDevice));
    k_to_bf16<<<nb(M.nparams), 256>>>(M.d_p, M.d_wb, (uint32_t)M.nparams);
    LSG_HIP(hipMemset(M.d_m, 0, 4 * M.nparams));
    LSG_HIP(hipMemset(M.d_v, 0, 4 * M.nparams));
    M.step = 0;
    LSG_HIP(hipDeviceSynchronize());
    return LSG_OK;
}

int lsg_mlp_get_params(const lsg_mlp* m, float* params)
{
    if (!m || !params) return fail(LSG_ERR_INVALID, "lsg_mlp_get_params: null argument");
    LSG_HIP(hipMemcpy(params, m->impl.d_p, 4 * m->impl.nparams, hipMemcpyDeviceToHost));
    return LSG_OK;
}

// x: device float[n x 32]; y: device float[n x 4]
int lsg_mlp_forward(lsg_mlp* m, const float* x, uint32_t n, float* y, void* stream)
{
    if (!m || (n && (!x || !y))) return fail(LSG_ERR_INVALID, "lsg_mlp_forward: null argument");
    MlpImpl& M = m->impl;
    hipStream_t s = (hipStream_t)stream;
    if (!n) return LSG_OK;
    MlpOffsets off;
    for (int l = 0; l < kLayers; l++) { off.w[l] = (uint32_t)M.wofs[l]; off.b[l] = (uint32_t)M.bofs[l]; }
    const uint64_t groups = ((uint64_t)n + 63) / 64;
    k_mlp_infer<<<(unsigned)std::min<uint64_t>(groups, kInferBlocks), 256, 0, s>>>(x, n, M.d_wb, M.d_p, off, y);
    LSG_HIP(hipGetLastError());
    return LSG_OK;
}

// one training step on n rows (n <= max_batch): forward, loss, backward, Adam.
// t: device float[n x 3] targets.  *loss (host) receives the mean loss when non-null
// (synchronises).  lr <= 0 computes gradients without updating (gradient checks).
int lsg_mlp_train_step(lsg_mlp* m, const float* x, const float* t, uint32_t n, float lambda, float lr, float* loss, void* stream)
{
    if (!m || !x || !t || !n) return fail(LSG_ERR_INVALID, "lsg_mlp_train_step: bad argument");
    MlpImpl& M = m->impl;
    if (n > M.max_batch) return fail(LSG_ERR_LIMIT, "lsg_mlp_train_step: n %u > max_batch %u", n, M.max_batch);
    hipStream_t s = (hipStream_t)stream;
    MlpOffsets off;
    for (int l = 0; l < kLayers; l++) { off.w[l] = (uint32_t)M.wofs[l]; off.b[l] = (uint32_t)M.bofs[l]; }
    const uint32_t parts = (uint32_t)std::min<uint64_t>(((uint64_t)n + kRows - 1) / kRows, kTrainBlocks);
    float* loss_part = M.d_part + (size_t)kTrainBlocks * M.nparams;
    k_mlp_train<<<parts, 256, 0, s>>>(x, t, n, lambda, M.d_wb, M.d_p, off, (uint32_t)M.nparams, M.d_part, loss_part);
    AdamArgs A{M.d_p, M.d_m, M.d_v, M.d_wb, M.d_mask, lr, 0.9f, 0.999f, 1e-8f, 1.f, 1.f};
    if (lr > 0) {
        M.step++;
        A.c1 = 1.f - powf(A.b1, (float)M.step); A.c2 = 1.f - powf(A.b2, (float)M.step);
    }
    k_mlp_update<<<(unsigned)((M.nparams + 63) / 64), 256, 0, s>>>(M.d_part, parts, (uint32_t)M.nparams, M.d_g, A, loss_part, M.d_loss);
    LSG_HIP(hipGetLastError());
    if (loss) {
        float l = 0;
        LSG_HIP(hipMemcpyAsync(&l, M.d_loss, 4, hipMemcpyDeviceToHost, s));
        LSG_HIP(hipStreamSynchronize(s));
        *loss = l / (float)n;
    }
    return LSG_OK;
}

int lsg_mlp_get_grads(const lsg_mlp* m, float* grads)
{
    if (!m || !grads) return fail(LSG_ERR_INVALID, "lsg_mlp_get_grads: null argument");
    LSG_HIP(hipMemcpy(grads, m->impl.d_g, 4 * m->impl.nparams, hipMemcpyDeviceToHost));
    return LSG_OK;
}

// verification hook: C[MxN] = A[MxK] B[KxN] with bf16 row-major inputs on the device, by
// k_gemm_bf16 (M, N, K multiples of 16)
int lsg_mlp_gemm_test(const uint16_t* A, const uint16_t* B, float* C, uint32_t M, uint32_t N, uint32_t K)
{
    if (!A || !B || !C || !M || !N || !K || M % 16 || N % 16 || K % 16) return fail(LSG_ERR_INVALID, "gemm_test: bad shape");
    k_gemm_bf16<<<(unsigned)((uint64_t)(M / 16) * (N / 16) + 3) / 4, 256>>>(A, B, C, (int)M, (int)N, (int)K);
    LSG_HIP(hipGetLastError());
    LSG_HIP(hipDeviceSynchronize());
    return LSG_OK;
}

} // extern "C"
