// lsgpu_encode.hip -- a filtered lightmap written into a consumer buffer's format on the GPU
// (gfx950), so a caller downloads 1-16 bytes per texel instead of the 16-byte work texel.
//
// The conversion is the last step of RRSolver::updateLightmap for a pixel buffer
// (lightmap.cpp:866-876) as the reference performs it through its buffer interface:
//   lightmapFillBackground (RRBuffer.cpp:964-975): a texel with alpha <= 0 takes the
//     background colour, made linear first (toLinear) when the target is scaled and the
//     solver has a colour space;
//   copyElementsTo (RRBuffer.cpp:105-131) from the linear work buffer: rgb to the target's
//     colour space (fromLinear) when the target is scaled;
//   RRBufferInMemory::setElement (RRBufferInMemory.cpp:229-285): integer formats take
//     RR_FLOAT2BYTE(x) = clamp(int(x * 256), 0, 255) (RRMath.h:78), luminance the rgb average
//     (x + y + z) * 0.33333333333333f, float formats the values.
// The colour space is the reference's sRGB approximation (RRGammaScaler, RRColorSpace.cpp:
// 22-91): x -> sign(x) |x|^gamma, evaluated as the reference's build does, in binary64
// rounded to binary32.  int(x * 256) follows x86-64's conversion, which gives INT_MIN (so 0
// after the clamp) for a product outside the int range or NaN.
#include "lsgpu_internal.h"
#include <cmath>

namespace lsg {
namespace {

__device__ inline float gamma_pow(float x, float g)
{
    return x >= 0.f ? (float)pow((double)x, (double)g) : -(float)pow((double)-x, (double)g);
}

__device__ inline uint32_t to_byte(float f)
{
    const float p = f * 256.f;
    const int v = (p >= -2147483648.f && p < 2147483648.f) ? (int)p : (int)0x80000000u;
    return (uint32_t)(v < 0 ? 0 : (v > 255 ? 255 : v));
}

// to_byte(gamma_pow(x, g)), for byte formats.  The power in binary32 decides the byte unless it
// falls within 2^-10 of where bytes change: with y = g log2 x its error is at most |y| 2^-22 (two
// functions good to an ulp and a product), so 256 * 2^y is off by at most 256 ln2 |y| 2^y 2^-22
// < 2^-15, whatever g.  The other few (1 in 500, and anything negative, infinite or NaN) take
// the binary64 power; it alone bound the kernel: 3.7M texels to RGB bytes 99 -> 54 us, half of it this.
__device__ inline uint32_t gamma_byte(float x, float g)
{
    if (x == 0.f && g > 0.f) return 0u;
    const float p = exp2f(g * log2f(x)) * 256.f, f = floorf(p), r = p - f;
    constexpr float kNear = 0x1p-10f;
    if (p < 300.f && (f >= 255.f ? p > 255.f + kNear : (r > kNear && r < 1.f - kNear))) return f < 255.f ? (uint32_t)f : 255u;
    return to_byte(gamma_pow(x, g));
}

struct EncodeArgs {
    const float4* rgba;
    uint32_t n;
    int32_t format;
    int32_t convert;        // rgb to the target's colour space
    float gamma;
    float4 bg;              // background, already as the fill uses it
    void* out;
};

// 1024 texels per workgroup, one per lane and turn, so that a wave reads consecutive texels (four
// consecutive ones per lane take four times the cache lookups: 3.7M texels to RGB bytes 89 us ->
// 54 us, the bytes moved taking 15).  Formats of
// other than 4 bytes' multiples are put together in LDS and stored as whole 32-bit words.
constexpr uint32_t kEncodeTexels = 1024;

__global__ __launch_bounds__(256) void k_encode(EncodeArgs A)
{
    __shared__ uint32_t words[kEncodeTexels * 3 / 4];
    uint8_t* const bytes = (uint8_t*)words;
    const uint32_t base = blockIdx.x * kEncodeTexels, count = min(kEncodeTexels, A.n - base);
    const bool bgr = A.format == LSG_FORMAT_BGR;
    const bool packed = A.format == LSG_FORMAT_RGB || bgr || A.format == LSG_FORMAT_LUMINANCE;
    for (uint32_t j = threadIdx.x; j < count; j += 256) {
        const size_t i = (size_t)base + j;
        float4 c = A.rgba[i];
        if (c.w <= 0.f) c = A.bg;
        auto byte = [&](float x) { return A.convert ? gamma_byte(x, A.gamma) : to_byte(x); };     // a colour component
        if (packed && A.format != LSG_FORMAT_LUMINANCE) {
            const uint32_t r = byte(c.x), g = byte(c.y), b = byte(c.z);
            bytes[3 * j] = (uint8_t)(bgr ? b : r); bytes[3 * j + 1] = (uint8_t)g; bytes[3 * j + 2] = (uint8_t)(bgr ? r : b);
            continue;
        }
        if (A.format == LSG_FORMAT_RGBA) {
            ((uint32_t*)A.out)[i] = byte(c.x) | byte(c.y) << 8 | byte(c.z) << 16 | to_byte(c.w) << 24;
            continue;
        }
        if (A.convert) { c.x = gamma_pow(c.x, A.gamma); c.y = gamma_pow(c.y, A.gamma); c.z = gamma_pow(c.z, A.gamma); }
        const float lum = (c.x + c.y + c.z) * 0.33333333333333f;
        switch (A.format) {
        case LSG_FORMAT_RGBF: {
            float* o = (float*)A.out + 3 * i;
            o[0] = c.x; o[1] = c.y; o[2] = c.z;
            break;
        }
        case LSG_FORMAT_RGBAF: ((float4*)A.out)[i] = c; break;
        case LSG_FORMAT_LUMINANCE: bytes[j] = (uint8_t)to_byte(lum); break;
        case LSG_FORMAT_LUMINANCEF: ((float*)A.out)[i] = lum; break;
        default: break;
        }
    }
    if (!packed) return;
    __syncthreads();
    const uint32_t size = A.format == LSG_FORMAT_LUMINANCE ? 1u : 3u, nbytes = count * size;
    uint8_t* const o = (uint8_t*)A.out + (size_t)base * size;
    for (uint32_t k = threadIdx.x; k < (nbytes + 3) / 4; k += 256) {
        if (4 * k + 4 <= nbytes) ((uint32_t*)o)[k] = words[k];
        else for (uint32_t q = 4 * k; q < nbytes; q++) o[q] = bytes[q];
    }
}

} // namespace
} // namespace lsg

using namespace lsg;

extern "C" {

uint32_t lsg_format_bytes(int32_t format)
{
    switch (format) {
    case LSG_FORMAT_RGB: case LSG_FORMAT_BGR: return 3;
    case LSG_FORMAT_RGBA: return 4;
    case LSG_FORMAT_RGBF: return 12;
    case LSG_FORMAT_RGBAF: return 16;
    case LSG_FORMAT_LUMINANCE: return 1;
    case LSG_FORMAT_LUMINANCEF: return 4;
    default: return 0;
    }
}

int lsg_lightmap_encode(const float* rgba, uint32_t ntexels, int32_t format, int32_t scaled, float solver_gamma, float copy_gamma,
                        const float* background, void* out, void* stream)
{
    if (!rgba || !out || !background) return fail(LSG_ERR_INVALID, "lsg_lightmap_encode: null argument");
    if (!lsg_format_bytes(format)) return fail(LSG_ERR_INVALID, "lsg_lightmap_encode: format %d has no per-texel encoding", format);
    const bool byte3 = format == LSG_FORMAT_RGB || format == LSG_FORMAT_BGR, word = format == LSG_FORMAT_RGBA;
    if ((byte3 || word || format == LSG_FORMAT_LUMINANCE) && ((uintptr_t)out & 3u))
        return fail(LSG_ERR_INVALID, "lsg_lightmap_encode: output must be 4-byte aligned");
    if (!ntexels) return LSG_OK;
    EncodeArgs A;
    A.rgba = (const float4*)rgba; A.n = ntexels; A.format = format; A.out = out;
    A.convert = scaled && copy_gamma > 0.f;
    A.gamma = copy_gamma;
    float bg[4] = {background[0], background[1], background[2], background[3]};
    if (scaled && solver_gamma > 0.f) {
        const float inv = 1 / solver_gamma;          // RRGammaScaler keeps 1/gamma in binary32
        for (int k = 0; k < 3; k++)
            bg[k] = bg[k] >= 0 ? (float)std::pow((double)bg[k], (double)inv) : -(float)std::pow((double)-bg[k], (double)inv);
    }
    A.bg = make_float4(bg[0], bg[1], bg[2], bg[3]);
    k_encode<<<ntexels / kEncodeTexels + (ntexels % kEncodeTexels ? 1u : 0u), 256, 0, (hipStream_t)stream>>>(A);
    LSG_HIP(hipGetLastError());
    return LSG_OK;
}

} // extern "C"
