/*
 * denoise.h - the denoise step of a render (the reference runs Intel Open Image Denoise on the host,
 * VulkanRendererPathTracing.cpp:985-1018, with the radiance, albedo and normal images).
 *
 * This library's own filter, on the GPU: an edge-avoiding a-trous wavelet filter (Dammertz, Sewtz, Hanika and
 * Lensch, "Edge-Avoiding A-Trous Wavelet Transform for fast Global Illumination Filtering", HPG 2010) over the
 * albedo-demodulated radiance, with edge-stopping weights from the normal and albedo AOVs and from the filtered
 * signal itself, then remodulated by the albedo.
 */
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>

namespace vvpt {

constexpr int kDenoiseLevels = 5;         /* a-trous steps 1, 2, 4, 8, 16 pixels: a 125-pixel footprint */
constexpr float kDenoiseSigmaColor = 0.5f;  /* on log(1 + irradiance), per channel */
constexpr float kDenoiseSigmaAlbedo = 0.02f; /* surfaces whose albedo differs by more do not mix (an emitter and
                                                the ceiling around it: 0.78 vs 0.73) */
constexpr float kDenoiseNormalPower = 64.0f;

/* Denoises W x H RGBA float images (device pointers; the normal in the AOV encoding n * 0.5 + 0.5).  tmp holds
 * 2 * W * H float4.  out may be any of the inputs.  Returns an error message or "". */
std::string denoise_device(const float *radiance, const float *albedo, const float *normal, uint32_t W, uint32_t H,
                           float *out, float *tmp, hipStream_t stream);

/* Largest image (pixels) of the allocation-free denoise: its two ping-pong images live in a fixed device array of
 * 2 * kDenoiseScratchPixels float4 (64 MiB per GPU the library runs on, held until the process ends). */
constexpr uint32_t kDenoiseScratchPixels = 1u << 21; /* 2,097,152 >= 1920 x 1080 */

/* Looks up the device address of that array on the current device `device` (once per device; later calls return
 * at once).  Returns an error message or "". */
std::string denoise_scratch_init(int device);

/* denoise_device with the fixed array as its scratch on `device` (denoise_scratch_init must have succeeded there):
 * allocates nothing, launches on `stream` and returns without waiting.  Every call on one GPU uses the same array,
 * so calls that overlap on that GPU (on different streams) race. */
std::string denoise_device_noalloc(const float *radiance, const float *albedo, const float *normal, uint32_t W,
                                   uint32_t H, float *out, int device, hipStream_t stream);

}  // namespace vvpt
