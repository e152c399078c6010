/*
 * denoise.hip - edge-avoiding a-trous filter on gfx950 (denoise.h).
 *
 *   k_dn_level   one level: 5 x 5 taps of the B3-spline kernel (1/16, 1/4, 3/8, 1/4, 1/16) spaced `step`
 *                pixels apart, each weighted by exp(-|log(1 + c_q) - log(1 + c_p)|^2 / sigma_c^2) (relative
 *                differences, so an emitter does not bleed into its surroundings; sigma_c halves per level),
 *                max(0, n_p . n_q)^64 and exp(-|a_q - a_p|^2 / sigma_a^2); taps outside the image are skipped
 *                and the weights renormalised.  The first level divides the radiance by the albedo per channel
 *                (albedo below 1e-3 counts as 1), so texture detail is not blurred and the filter runs on what the
 *                albedo multiplies; the last multiplies it back, alpha 1.
 *
 * A block filters 16 x 16 pixels of one residue class (x mod step, y mod step), whose taps are each other's neighbours:
 * the 20 x 20 pixels they need are read, their logarithms taken and their normals decoded once, into LDS, instead of 25
 * times per pixel.  The step's step^2 classes of one image region are consecutive blocks of one die, so that the
 * interleaved lines they read are shared in its L2.  Bound by instruction issue (25 taps of about 45 instructions per
 * pixel).  1920 x 1080: the whole filter 0.374 ms instead of 2.44 (under a kernel trace 82 to 100 us a level, 571 before).
 */
#include "denoise.h"

#include <algorithm>
#include <mutex>
#include <vector>

/* Scratch of the allocation-free entry point: two ping-pong images of up to kDenoiseScratchPixels pixels.  Host
 * code never uses this name as an address (on the host it is only a stand-in for the symbol); the device address
 * of each GPU's copy comes from hipGetSymbolAddress in denoise_scratch_init and is what the kernels receive. */
static __device__ __align__(256) float4 scratch[2 * (size_t)vvpt::kDenoiseScratchPixels];

namespace vvpt {
namespace {

std::mutex g_scratch_mutex;
std::vector<float4 *> g_scratch_ptr; /* device address of `scratch` on each device (index = HIP device), or null */

__device__ __forceinline__ float4 dn_compress(float4 c) {
    return make_float4(log1pf(fmaxf(c.x, 0.0f)), log1pf(fmaxf(c.y, 0.0f)), log1pf(fmaxf(c.z, 0.0f)), 0.0f);
}

__device__ __forceinline__ float dn_demod(float a) { return a > 1e-3f ? a : 1.0f; }

/* Decoded AOV normal and whether the pixel saw a surface (a miss stores no normal). */
__device__ __forceinline__ bool dn_normal(float4 e, float3 &n) {
    n = make_float3(e.x * 2.0f - 1.0f, e.y * 2.0f - 1.0f, e.z * 2.0f - 1.0f);
    const float l2 = n.x * n.x + n.y * n.y + n.z * n.z;
    if (!(l2 > 0.25f)) return false;
    const float r = rsqrtf(l2);
    n = make_float3(n.x * r, n.y * r, n.z * r);
    return true;
}

constexpr int kDnTile = 16, kDnHalo = kDnTile + 4; /* outputs and staged pixels of a block, per axis */

template <bool FIRST, bool LAST>
__global__ __launch_bounds__(kDnTile * kDnTile) void k_dn_level(const float4 *src, float4 *dst, const float4 *alb,
                                                                const float4 *nrm, uint32_t W, uint32_t H, int step,
                                                                uint32_t tiles_x, uint32_t nblocks, float inv_sc2) {
    /* a staged pixel: (c, t.x), (t.y, t.z, a.x, a.y), (a.z, n); n = 0 where the pixel saw no surface, and NaN outside the
     * image, which is a zero weight against pixels with and without one */
    __shared__ float4 tile[3][kDnHalo * kDnHalo];
    /* the blocks of one die (block % 8) take consecutive (tile, y class, x class) triples */
    const uint32_t per = (nblocks + 7u) / 8u, lin = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    if (lin >= nblocks) return;
    const uint32_t cx = min((uint32_t)step, W), cy = min((uint32_t)step, H); /* classes that hold a pixel */
    const uint32_t rx = lin % cx, ry = lin / cx % cy, tl = lin / (cx * cy);
    const int tx = (int)(tl % tiles_x) * kDnTile, ty = (int)(tl / tiles_x) * kDnTile; /* in pixels of the class */
    const int lx = threadIdx.x, ly = threadIdx.y;
    for (int k = ly * kDnTile + lx; k < kDnHalo * kDnHalo; k += kDnTile * kDnTile) {
        const int qx = (tx + k % kDnHalo - 2) * step + (int)rx, qy = (ty + k / kDnHalo - 2) * step + (int)ry;
        float4 c = make_float4(0.f, 0.f, 0.f, 0.f), t = c, a = c;
        float3 n = make_float3(NAN, NAN, NAN);
        if (qx >= 0 && qx < (int)W && qy >= 0 && qy < (int)H) {
            const size_t q = (size_t)qy * W + qx;
            c = src[q];
            a = alb[q];
            if (FIRST) c = make_float4(c.x / dn_demod(a.x), c.y / dn_demod(a.y), c.z / dn_demod(a.z), 0.0f);
            t = dn_compress(c);
            if (!dn_normal(nrm[q], n)) n = make_float3(0.f, 0.f, 0.f);
        }
        tile[0][k] = make_float4(c.x, c.y, c.z, t.x);
        tile[1][k] = make_float4(t.y, t.z, a.x, a.y);
        tile[2][k] = make_float4(a.z, n.x, n.y, n.z);
    }
    __syncthreads();
    const int x = (tx + lx) * step + (int)rx, y = (ty + ly) * step + (int)ry;
    if (x >= (int)W || y >= (int)H) return;
    const float h[5] = {1.0f / 16.0f, 1.0f / 4.0f, 3.0f / 8.0f, 1.0f / 4.0f, 1.0f / 16.0f};
    const int centre = (ly + 2) * kDnHalo + lx + 2;
    const float4 p0 = tile[0][centre], p1 = tile[1][centre], p2 = tile[2][centre];
    const bool sp = p2.y != 0.0f || p2.z != 0.0f || p2.w != 0.0f;
    const float inv_sa2 = 1.0f / (kDenoiseSigmaAlbedo * kDenoiseSigmaAlbedo);
    float4 sum = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float wsum = 0.0f;
#pragma unroll 1 /* a row's taps in flight: all 25 unrolled hold 258 registers */
    for (int j = 0; j < 5; ++j) {
        const float hj = j == 2 ? 3.0f / 8.0f : ((j & 1) ? 1.0f / 4.0f : 1.0f / 16.0f);
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            const int k = (ly + j) * kDnHalo + lx + i;
            const float4 q0 = tile[0][k], q1 = tile[1][k], q2 = tile[2][k];
            const float dx = q0.w - p0.w, dy = q1.x - p1.x, dz = q1.y - p1.y;
            const float ax = q1.z - p1.z, ay = q1.w - p1.w, az = q2.x - p2.x;
            const float dc = dx * dx + dy * dy + dz * dz, da = ax * ax + ay * ay + az * az;
            float wn;
            if (sp) { /* 0 against a pixel without a surface or outside (fmaxf takes the number of a number and NaN) */
                wn = fmaxf(p2.y * q2.y + p2.z * q2.z + p2.w * q2.w, 0.0f);
                static_assert(kDenoiseNormalPower == 64.0f, "six squarings");
#pragma unroll
                for (int e = 0; e < 6; ++e) wn *= wn;
            } else {
                wn = (q2.y != 0.0f || q2.z != 0.0f || q2.w != 0.0f) ? 0.0f : 1.0f;
            }
            const float w = h[i] * hj * __expf(-dc * inv_sc2 - da * inv_sa2) * wn;
            sum.x += w * q0.x;
            sum.y += w * q0.y;
            sum.z += w * q0.z;
            wsum += w;
        }
    }
    /* the centre tap has weight h2 * h2 > 0, so wsum > 0 */
    const float r = 1.0f / wsum;
    const size_t p = (size_t)y * W + x;
    if (LAST)
        dst[p] = make_float4(sum.x * r * dn_demod(p1.z), sum.y * r * dn_demod(p1.w), sum.z * r * dn_demod(p2.x), 1.0f);
    else
        dst[p] = make_float4(sum.x * r, sum.y * r, sum.z * r, 0.0f);
}

}  // namespace

std::string denoise_device(const float *radiance, const float *albedo, const float *normal, uint32_t W, uint32_t H,
                           float *out, float *tmp, hipStream_t s) {
    /* Every level reads what the one before it wrote, the first the radiance, and its neighbours' albedo and normals; only
     * the last writes out.  out may be the radiance itself; where it shares memory with the albedo or the normals, which
     * other blocks of that level still read, the level goes to tmp and is copied. */
    const size_t bytes = (size_t)W * H * sizeof(float4);
    auto shares = [&](const float *in) { return (uintptr_t)in < (uintptr_t)out + bytes && (uintptr_t)out < (uintptr_t)in + bytes; };
    const bool copy = shares(albedo) || shares(normal);
    float4 *img[2] = {(float4 *)tmp, (float4 *)tmp + (size_t)W * H};
    const float4 *src = (const float4 *)radiance, *alb = (const float4 *)albedo, *nrm = (const float4 *)normal;
    float sc = kDenoiseSigmaColor;
    static_assert(kDenoiseLevels >= 2, "the first and the last level are different launches");
    for (int l = 0; l < kDenoiseLevels; ++l) {
        const uint32_t step = 1u << l;
        const uint32_t tiles_x = ((W + step - 1) / step + kDnTile - 1) / kDnTile;
        const uint32_t tiles_y = ((H + step - 1) / step + kDnTile - 1) / kDnTile;
        /* a strip has fewer classes than step * step; blocks of 16 x 16 keep the longest one (2^28 pixels) within the
         * 2^32 threads a launch may have per axis */
        const uint32_t nblocks = tiles_x * tiles_y * std::min(step, W) * std::min(step, H);
        const dim3 grid((nblocks + 7u) / 8u * 8u), blk(kDnTile, kDnTile);
        float4 *dst = l + 1 == kDenoiseLevels && !copy ? (float4 *)out : img[l & 1];
        const float inv_sc2 = 1.0f / (sc * sc);
        if (l == 0)
            hipLaunchKernelGGL((k_dn_level<true, false>), grid, blk, 0, s, src, dst, alb, nrm, W, H, (int)step, tiles_x, nblocks, inv_sc2);
        else if (l + 1 < kDenoiseLevels)
            hipLaunchKernelGGL((k_dn_level<false, false>), grid, blk, 0, s, src, dst, alb, nrm, W, H, (int)step, tiles_x, nblocks, inv_sc2);
        else
            hipLaunchKernelGGL((k_dn_level<false, true>), grid, blk, 0, s, src, dst, alb, nrm, W, H, (int)step, tiles_x, nblocks, inv_sc2);
        src = dst;
        sc *= 0.5f;
    }
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && copy) e = hipMemcpyAsync(out, src, bytes, hipMemcpyDeviceToDevice, s);
    return e == hipSuccess ? std::string() : std::string(hipGetErrorString(e));
}

std::string denoise_scratch_init(int device) {
    if (device < 0) return "invalid device";
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if ((size_t)device < g_scratch_ptr.size() && g_scratch_ptr[device]) return "";
    void *p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e);
    if (!p) return "hipGetSymbolAddress(scratch) returned no address";
    if ((size_t)device >= g_scratch_ptr.size()) g_scratch_ptr.resize((size_t)device + 1, nullptr);
    g_scratch_ptr[device] = (float4 *)p;
    return "";
}

std::string denoise_device_noalloc(const float *radiance, const float *albedo, const float *normal, uint32_t W,
                                   uint32_t H, float *out, int device, hipStream_t stream) {
    if ((uint64_t)W * H > kDenoiseScratchPixels)
        return "image of " + std::to_string((uint64_t)W * H) + " pixels exceeds the " +
               std::to_string(kDenoiseScratchPixels) + "-pixel scratch of the allocation-free denoise";
    float4 *tmp = nullptr;
    {
        std::lock_guard<std::mutex> lock(g_scratch_mutex);
        if (device >= 0 && (size_t)device < g_scratch_ptr.size()) tmp = g_scratch_ptr[device];
    }
    if (!tmp) return "no scratch address on this device";
    /* the first level writes every pixel of the first image and each level every pixel of the next before they are read:
     * nothing in the scratch needs to start at zero, and what a previous call left there is never read */
    return denoise_device(radiance, albedo, normal, W, H, out, (float *)tmp, stream);
}

}  // namespace vvpt
