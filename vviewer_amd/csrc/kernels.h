/*
 * kernels.h - wavefront path-tracing kernels for gfx950.
 *
 * The reference runs one raygen invocation per pixel that loops over the
 * batch's samples and bounces, with recursive traceRayEXT calls for shadow and
 * emitter-lookup rays (raygen.rgen.glsl:24-145, rayPrimary*.rchit.glsl).  Here
 * that loop is split into queues: a path slot owns one work item
 * (pixel, batch) at a time, runs its batchSize samples in order with the RNG
 * state carried across samples (rng_def.glsl:32-36, raygen.rgen.glsl:37,55), and
 * every iteration of the host loop advances all active slots by one bounce:
 *
 *   k_secondary  shadow segments and emitter-lookup walks of the previous bounce that need the general walk (any-hit
 *                logic applied closest-first)
 *   k_shadow     single-segment shadow rays of the previous bounce
 *   k_extend     closest-hit query of each slot's ray; when the previous bounce
 *                asked for a BSDF-direction emitter lookup (next_event_estimation.glsl)
 *                the same walk also answers it (MODE_CLOSEST2)
 *   k_shade      adds the previous bounce's secondary results in a fixed order, then one bounce of the closest-hit /
 *                miss shaders; light sampling and emitter lookups that need their own walk become records in a
 *                shadow or secondary queue; samples that end are accumulated, finished work items written and
 *                replaced, camera rays regenerated, and the next queue compacted (wave ballot + prefix count, one
 *                atomic per wave)
 *
 * Results of a work item depend only on (pixel, batch), so the image is the
 * same whatever the slot scheduling; k_resolve sums the per-batch partials in
 * batch order like the reference's per-batch image read-modify-write
 * (raygen.rgen.glsl:134-144).
 */
#pragma once
#include "env_sampling.h"
#include "queue.h"
#include "sampler.h"
#include "traverse.h"

namespace vvpt {

constexpr int kTraceBlock = 128;
/* k_extend and k_shadow: at least 5 waves per SIMD (at most 102 VGPRs; 4 otherwise) where the LDS stack allows it
 * (STACK <= 16).  Their walks wait on dependent node loads, so resident waves hide latency (k_shadow 116 -> 107 ms
 * per 1080p frame at 64 spp; k_extend 67.3 -> 62.4 ms once its world ray and saved TLAS position moved to LDS and it
 * fitted in 92 VGPRs without spilling); 6 waves would spill registers to scratch, and so would the counting k_extend
 * at 5. */
#define VVPT_TRACE_OCCUPANCY __attribute__((amdgpu_waves_per_eu(STACK <= 16 ? (COUNT ? 4 : 5) : 1, 8)))
constexpr int kBlock = 256;

enum : uint32_t {
    F_NEE = 1u,        /* the slot's ray also carries the previous bounce's emitter lookup */
    F_DONE = 2u,       /* the sample is over and waits for the results named by the other bits (parked) */
    F_SEC0 = 4u,       /* secondary record 0 (shadow ray) pending */
    F_SEC1 = 8u,       /* secondary record 1 (emitter lookup of the previous bounce) pending */
    F_SEC2 = 16u,      /* secondary record 2 (emitter lookup of the last bounce) pending */
    F_TERMINAL = 32u,  /* the ray only carries the last bounce's emitter lookup; the sample ends after it */
    F_TPASS = 64u,     /* secondary record 1 is the 1 - alpha product in front of a found emitter */
    F_NRCQ = 128u,     /* the path ended in a radiance-cache query (inputs in orig / dir / nee, weight in beta) */
    F_NRC_FALLBACK = 256u /* returned by shade_one only: the path would have ended in a query, but the cache's error
                             estimate there exceeds its tolerance, so it continues */
};

/* Extension-queue entries are slots; an entry with this bit set has no ray to trace: its sample is over but waits for
 * results still being computed (shadow records, a cache query), which the next k_shade adds before it ends it. */
constexpr uint32_t kParked = 0x80000000u;

/* stats[] slots (64-bit); each wave adds into the copy of its shard (kStatStride apart) */
enum : uint32_t {
    S_PATH = 0, S_SHADOW = 1, S_NEE = 2, S_NODES_EXT = 3, S_TRIS_EXT = 4, S_NODES_SEC = 5, S_TRIS_SEC = 6,
    S_NODES_SHD = 7, S_TRIS_SHD = 8, S_SHADOW_SEC = 9, S_NRCQ = 10, S_NRC_FALLBACK = 11, S_NSTATS = 12
};
constexpr uint32_t kStatStride = 16; /* 128 bytes of uint64 per shard */

/* Path-state arrays are streamed: each kernel of an iteration touches a slot's record once, and the records of
 * all slots (gigabytes) pass through the caches between two touches, so stores to them are non-temporal, which
 * leaves more of L2 to the shading data (instances, materials, vertices: megabytes, read by every bounce).  Loads
 * stay ordinary: lanes of neighbouring waves read neighbouring records, and non-temporal loads measured slower
 * (1080p icosphere field: ordinary 715.7, non-temporal stores 720.7, non-temporal loads and stores 706.6
 * Msamples/s).  st.x[i] reads and assignments go through StreamRef; element types and values are unchanged. */
template <class T>
struct StreamRef {
    T *p;
    __device__ __forceinline__ operator T() const { return *p; }
    __device__ __forceinline__ const StreamRef &operator=(T v) const {
        __builtin_nontemporal_store(v, p);
        return *this;
    }
};
typedef float v4f_t __attribute__((ext_vector_type(4)));
typedef float v2f_t __attribute__((ext_vector_type(2)));
template <>
struct StreamRef<float4> {
    float4 *p;
    __device__ __forceinline__ operator float4() const { return *p; }
    __device__ __forceinline__ const StreamRef &operator=(float4 a) const {
        const v4f_t v = {a.x, a.y, a.z, a.w};
        __builtin_nontemporal_store(v, reinterpret_cast<v4f_t *>(p));
        return *this;
    }
};
template <>
struct StreamRef<float2> {
    float2 *p;
    __device__ __forceinline__ operator float2() const { return *p; }
    __device__ __forceinline__ const StreamRef &operator=(float2 a) const {
        const v2f_t v = {a.x, a.y};
        __builtin_nontemporal_store(v, reinterpret_cast<v2f_t *>(p));
        return *this;
    }
};
template <class T>
struct StreamArray {
    T *p;
    __host__ __device__ StreamArray &operator=(T *q) {
        p = q;
        return *this;
    }
    __device__ __forceinline__ StreamRef<T> operator[](uint32_t i) const { return StreamRef<T>{p + i}; }
};

struct PathState {
    StreamArray<uint32_t> item, rng, ctr, vol, flags;
    StreamArray<uint32_t> job; /* batched render: the slot's job */
    StreamArray<float4> orig, dir, beta, nee, L, accR, accA, accN, payA, payN;
    /* k_extend's answer, one 64-byte record per slot (4 s .. 4 s + 3), so that a finished walk writes whole 32-byte
     * sectors of one line instead of parts of five arrays: [0] the path hit (t, u, v, prim); [1] its instance, the
     * emitter lookup's instance and the nearest candidate that lookup passed; [2] the lookup's hit (t, u, v, prim)
     * and [3] zero, written only with a lookup */
    StreamArray<float4> hit;
    /* secondary records, 3 per slot, stored planar: record k of slot s at k * nsec + s (sec_ix), so the records
     * of neighbouring slots are neighbours; queues carry the record as 3 s + k */
    StreamArray<float4> sec_o, sec_d, sec_c;
    StreamArray<uint32_t> sec_v;
    uint32_t nsec;
    /* radiance cache (extended mode with the cache on) */
    StreamArray<uint32_t> nrct; /* training-record block of the current sample, or kInvalid */
    StreamArray<float2> spread; /* path spread: x = footprint of the primary vertex, y = sum of sqrt(area) after it */
};

struct RenderParams {
    uint32_t items_total; /* work items of this launch window (all jobs) */
    uint32_t aovs;
    uint32_t media;    /* a path can be inside a medium (Features::vol): the slots' volumes are kept */
    uint32_t nslots;
    float total_samples;
    SQueue ext[2]; /* slots with a ray to extend (double-buffered across iterations) */
    SQueue sec;    /* secondary records needing a general walk (3 per slot) */
    SQueue shd;    /* single-segment shadow rays (scenes without volume-changing surfaces) */
    uint32_t *items; /* kShards padded work-item counters */
    uint32_t items_per_shard;
    uint32_t item_chunk; /* 0: contiguous item shards; else chunks of this many items dealt round-robin */
    unsigned long long *stats; /* kShards * kStatStride */
    float4 *partR, *partA, *partN;
    /* radiance cache */
    uint32_t nrc;              /* the cache is trained on this render's paths */
    uint32_t nrc_use;          /* paths may end in cache queries */
    uint32_t nrc_vmax;         /* vertices recorded per training sample */
    uint32_t nrc_thresh;       /* a sample trains the cache when its hash is below this */
    float nrc_c;               /* spread threshold: query once spread^2 > c * footprint */
    uint32_t *nrc_ctr;         /* [0] training blocks taken, [1] training samples written, [2] queries */
    uint32_t nrc_blocks;       /* training blocks available */
    float *nrc_pool;           /* training blocks: nrc_vmax vertices x 16 floats (input 10, L before 3, beta 3) */
    float *nrc_tin, *nrc_ttgt; /* training samples: inputs (10 floats) and targets (3 floats) */
    uint32_t nrc_tcap;
    SQueue nrcq;               /* slots that ended in a cache query this iteration */
    float *nrc_qin;            /* gathered query inputs (10 floats each) */
    uint32_t *nrc_qslot;
    float *nrc_qpred;          /* predictions (3 floats each) */
    const uint8_t *nrc_ok;     /* cells of the error grid where the cache may answer queries (null: everywhere) */
    float nrc_lo[3], nrc_cells[3]; /* world position -> error-grid cell: (p - lo) * cells, per axis */
};

/* The cache's error estimate at a world position is within its tolerance (nrc.h kNrcErrRes grid; the flags come
 * from the training samples of earlier frames, k_nrc_err_flags).  Elsewhere the path goes on without the cache:
 * the plain (extended) estimator is the fallback. */
__device__ __forceinline__ bool nrc_region_ok(const RenderParams &P, f3 wp) {
    if (!P.nrc_ok) return true;
    const float q[3] = {wp.x, wp.y, wp.z};
    uint32_t c[3];
    for (int a = 0; a < 3; ++a)
        c[a] = min((uint32_t)fmaxf((q[a] - P.nrc_lo[a]) * P.nrc_cells[a], 0.0f), kNrcErrRes - 1u);
    return P.nrc_ok[c[0] + kNrcErrRes * (c[1] + kNrcErrRes * c[2])] != 0u;
}

/* ctr word: sample (bits 0..15) | depth d (16..23) | surfaceDepth (24..31) */
__device__ __forceinline__ uint32_t ctr_sample(uint32_t c) { return c & 0xffffu; }
__device__ __forceinline__ uint32_t ctr_depth(uint32_t c) { return (c >> 16) & 0xffu; }
__device__ __forceinline__ uint32_t ctr_sdepth(uint32_t c) { return c >> 24; }
__device__ __forceinline__ uint32_t ctr_make(uint32_t s, uint32_t d, uint32_t sd) {
    return (s & 0xffffu) | ((d & 0xffu) << 16) | (sd << 24);
}

__device__ __forceinline__ uint32_t lane_id() { return __lane_id(); }

/* Random numbers of one path sample: the reference's xorshift stream in parity mode (rng_def.glsl:4-36; s is the
 * state, carried across the samples of a batch), the scrambled Sobol points of sampler.h in the extended mode (s is
 * the next dimension, n the sample index within the pixel, key the pixel's sequence key). */
struct Rng {
    uint32_t s, n, key;
    bool ld;
};
__device__ __forceinline__ float rnd(Rng &r) {
    if (r.ld) return sampler_float(r.key, r.n, r.s++);
    return rand1D(r.s);
}
/* The job of a path slot (the kernel argument in a single render). */
template <bool MULTI>
__device__ __forceinline__ const JobView &job_of(const DScene &S, const PathState &st, uint32_t slot) {
    if (MULTI) return S.jobs[st.job[slot]];
    return S.job;
}

/* Job of a global work item of a batched render: binary search over the jobs' first items. */
__device__ __forceinline__ uint32_t job_of_item(const DScene &S, uint32_t item) {
    uint32_t lo = 0, hi = S.njobs;
    while (hi - lo > 1u) {
        const uint32_t mid = (lo + hi) >> 1;
        if (S.jobs[mid].item_begin <= item) lo = mid; else hi = mid;
    }
    return lo;
}

/* Training samples of a finished training path: the radiance leaving each recorded vertex towards the previous
 * one is (L_final - L_before) / throughput, component-wise (Müller et al. 2021: the suffix's own estimate). */
__device__ __forceinline__ void nrc_emit_training(const RenderParams &P, uint32_t tb, uint32_t nv, f3 Lf) {
    if (nv == 0u) return;
    const uint32_t base = atomicAdd(P.nrc_ctr + 1, nv);
    for (uint32_t v = 0; v < nv && base + v < P.nrc_tcap; ++v) {
        const float *r = P.nrc_pool + ((size_t)tb * P.nrc_vmax + v) * 16u;
        float *in = P.nrc_tin + (size_t)(base + v) * 10u;
        for (int k = 0; k < 10; ++k) in[k] = r[k];
        const float Lb[3] = {r[10], r[11], r[12]}, b[3] = {r[13], r[14], r[15]}, lf[3] = {Lf.x, Lf.y, Lf.z};
        float *t = P.nrc_ttgt + (size_t)(base + v) * 3u;
        for (int c = 0; c < 3; ++c) t[c] = b[c] > 1e-8f ? fmaxf(lf[c] - Lb[c], 0.0f) / b[c] : 0.0f;
    }
}

/* Radiance-cache state of a starting sample: a small hashed fraction of samples trains the cache (their paths
 * are traced to the end and every surface vertex is recorded), the others may end in a cache query. */
__device__ __forceinline__ void nrc_sample_start(const RenderParams &P, const JobView &J, const PathState &st, uint32_t slot,
                                                 uint32_t item, uint32_t sample) {
    uint32_t t = kInvalid;
    const uint32_t bl = item / J.npix, pix = item - bl * J.npix;
    const uint32_t h = hash_mix(sampler_key(pix, J.seed ^ 0x2545f491u), (J.batch_begin + bl) * J.batch_size + sample);
    if (h < P.nrc_thresh) {
        const uint32_t b = atomicAdd(P.nrc_ctr, 1u);
        if (b < P.nrc_blocks) t = b;
    }
    st.nrct[slot] = t;
    st.spread[slot] = make_float2(0.0f, 0.0f);
}

/* What a render can meet, fixed when k_shade is compiled: a kernel that carries every estimator's code for every
 * scene is 170 KB of instructions (more than the instruction cache of two CUs) and keeps its kernel arguments in
 * spilled registers. */
template <bool EXT_, bool NRC_, bool TEX_, bool VOL_>
struct Features {
    static constexpr bool ext = EXT_; /* the extended estimator (scrambled Sobol samples, environment sampling) */
    static constexpr bool nrc = NRC_; /* the radiance cache (with ext) */
    static constexpr bool tex = TEX_; /* some surface has a texture of its own besides the alpha cut-out */
    static constexpr bool vol = VOL_; /* a path can be inside a medium: the camera is, or a surface bounds one */
};

/* Generator of sample `sample` of the job's work item `item` (parity: the stored xorshift state). */
template <class Fx>
__device__ __forceinline__ Rng rng_of(const JobView &J, uint32_t state, uint32_t item, uint32_t sample) {
    Rng r;
    r.s = state;
    r.ld = Fx::ext;
    r.n = 0u;
    r.key = 0u;
    if (r.ld) {
        const uint32_t bl = item / J.npix, pix = item - bl * J.npix;
        r.n = (J.batch_begin + bl) * J.batch_size + sample;
        r.key = sampler_key(pix, J.seed);
    }
    return r;
}

/* Wave-aggregated append: one atomic per wave.  Every lane of the wave must call it. */
__device__ __forceinline__ uint32_t wave_append(uint32_t *counter, bool pred) {
    const unsigned long long mask = __ballot(pred);
    const uint32_t lane = lane_id();
    const uint32_t prefix = __popcll(mask & ((1ull << lane) - 1ull));
    uint32_t base = 0;
    if (mask != 0ull) {
        const int leader = __ffsll((long long)mask) - 1;
        if ((int)lane == leader) base = atomicAdd(counter, (uint32_t)__popcll(mask));
        base = __shfl(base, leader);
    }
    return base + prefix;
}

/* Wave-aggregated append of n (0..3) entries per lane; returns the lane's first index. */
__device__ __forceinline__ uint32_t wave_append_n(uint32_t *counter, uint32_t n) {
    const unsigned long long m0 = __ballot((n & 1u) != 0u), m1 = __ballot((n & 2u) != 0u);
    const uint32_t lane = lane_id();
    const unsigned long long lt = (1ull << lane) - 1ull;
    const uint32_t prefix = __popcll(m0 & lt) + 2u * __popcll(m1 & lt);
    const uint32_t total = __popcll(m0) + 2u * __popcll(m1);
    uint32_t base = 0;
    if (total) {
        if (lane == 0) base = atomicAdd(counter, total);
        base = __shfl(base, 0);
    }
    return base + prefix;
}

__device__ __forceinline__ uint32_t wave_global_id() { return (blockIdx.x * blockDim.x + threadIdx.x) >> 6; }

/* Reduce v across the wave and add it to stat k of the wave's shard copy. */
__device__ __forceinline__ void wave_add64(unsigned long long *stats, uint32_t k, uint32_t v) {
    uint32_t s = v;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (lane_id() == 0 && s) atomicAdd(stats + (wave_global_id() % kShards) * kStatStride + k, (unsigned long long)s);
}

/* ------------------------------------------------------------- textures -- */
__device__ __forceinline__ float4 texel(const DScene &S, const DTexture &T, uint32_t x, uint32_t y) {
    const size_t k = (size_t)T.offset + (size_t)y * T.width + x;
    if (T.format == 2u) return S.texf[k];
    const uint32_t c = S.tex8[k];
    const float a = (float)(c >> 24) / 255.0f;
    if (T.format == 1u)
        return make_float4(S.srgb_lut[c & 0xffu], S.srgb_lut[(c >> 8) & 0xffu], S.srgb_lut[(c >> 16) & 0xffu], a);
    return make_float4((float)(c & 0xffu) / 255.0f, (float)((c >> 8) & 0xffu) / 255.0f,
                       (float)((c >> 16) & 0xffu) / 255.0f, a);
}
__device__ __forceinline__ uint32_t wrapi(int i, uint32_t n) {
    int m = i % (int)n;
    return (uint32_t)(m < 0 ? m + (int)n : m);
}
/* bilinear, repeat, LOD 0 (VulkanTexture.cpp:221-224) */
__device__ __forceinline__ float4 tex_sample(const DScene &S, uint32_t t, float u, float v) {
    const DTexture T = S.texs[t];
    if (T.width == 1u && T.height == 1u) return texel(S, T, 0, 0);
    const float x = u * (float)T.width - 0.5f, y = v * (float)T.height - 0.5f;
    const float fx = floorf(x), fy = floorf(y);
    const float a = x - fx, b = y - fy;
    const int ix = (int)fx, iy = (int)fy;
    const uint32_t x0 = wrapi(ix, T.width), x1 = wrapi(ix + 1, T.width);
    const uint32_t y0 = wrapi(iy, T.height), y1 = wrapi(iy + 1, T.height);
    const float4 t00 = texel(S, T, x0, y0), t10 = texel(S, T, x1, y0), t01 = texel(S, T, x0, y1),
                 t11 = texel(S, T, x1, y1);
    const float w00 = (1.0f - a) * (1.0f - b), w10 = a * (1.0f - b), w01 = (1.0f - a) * b, w11 = a * b;
    return make_float4(t00.x * w00 + t10.x * w10 + t01.x * w01 + t11.x * w11,
                       t00.y * w00 + t10.y * w10 + t01.y * w01 + t11.y * w11,
                       t00.z * w00 + t10.z * w10 + t01.z * w01 + t11.z * w11,
                       t00.w * w00 + t10.w * w10 + t01.w * w01 + t11.w * w11);
}
__device__ __forceinline__ f3 tex_rgb(const DScene &S, uint32_t t, float u, float v) {
    float4 c = tex_sample(S, t, u, v);
    return {c.x, c.y, c.z};
}

/* Equirect environment resampled to a cube map (VulkanRendererSkybox.cpp:98-140),
 * looked up with textureLod(skybox, dir, 0) (rayPrimary.rmiss.glsl:76). */
__device__ __forceinline__ f3 env_lookup(const DScene &S, f3 d) {
    if (S.cube_w == 0u) return {0, 0, 0};
    const float ax = fabsf(d.x), ay = fabsf(d.y), az = fabsf(d.z);
    int face;
    float sc, tc, ma;
    if (ax >= ay && ax >= az) {
        ma = ax;
        if (d.x > 0) { face = 0; sc = -d.z; tc = -d.y; } else { face = 1; sc = d.z; tc = -d.y; }
    } else if (ay >= az) {
        ma = ay;
        if (d.y > 0) { face = 2; sc = d.x; tc = d.z; } else { face = 3; sc = d.x; tc = -d.z; }
    } else {
        ma = az;
        if (d.z > 0) { face = 4; sc = d.x; tc = -d.y; } else { face = 5; sc = -d.x; tc = -d.y; }
    }
    const float s = 0.5f * (sc / ma + 1.0f), t = 0.5f * (tc / ma + 1.0f);
    const uint32_t w = S.cube_w;
    const float x = s * (float)w - 0.5f, y = t * (float)w - 0.5f;
    const float fx = floorf(x), fy = floorf(y);
    const float a = x - fx, b = y - fy;
    const float wm = (float)(w - 1);
    const uint32_t x0 = (uint32_t)fminf(fmaxf(fx, 0.0f), wm), x1 = (uint32_t)fminf(fmaxf(fx + 1.0f, 0.0f), wm);
    const uint32_t y0 = (uint32_t)fminf(fmaxf(fy, 0.0f), wm), y1 = (uint32_t)fminf(fmaxf(fy + 1.0f, 0.0f), wm);
    const float4 *F = S.cube + (size_t)face * w * w;
    const float4 c00 = F[y0 * w + x0], c10 = F[y0 * w + x1], c01 = F[y1 * w + x0], c11 = F[y1 * w + x1];
    const float w00 = (1 - a) * (1 - b), w10 = a * (1 - b), w01 = (1 - a) * b, w11 = a * b;
    return {c00.x * w00 + c10.x * w10 + c01.x * w01 + c11.x * w11, c00.y * w00 + c10.y * w10 + c01.y * w01 + c11.y * w11,
            c00.z * w00 + c10.z * w10 + c01.z * w01 + c11.z * w11};
}

/* ---------------------------------------- environment importance sampling -- */
/* Extended mode only (the reference never samples the environment, lightSampling.glsl:101-106): a grid of
 * env_mw x env_mh cells in (phi, theta) (theta from +y, phi = atan2(z, x)) with an alias table over the cells.
 * The cell weights bound the environment's radiance from above (k_env_importance), so the density covers every
 * direction with radiance.  A sample picks a cell (one uniform for the cell, one for the alias choice) and a
 * uniform point in it; its solid-angle density is p_cell * cells / (2 pi^2 sin theta). */
__device__ __forceinline__ f3 env_dir_of(float phi, float theta) {
    f3 d;
    env_dir(phi, theta, d.x, d.y, d.z);
    return d;
}

__device__ __forceinline__ float env_pdf_dir(const DScene &S, f3 d) {
    return env_pdf(S.env_cpdf, S.env_mw, S.env_mh, d.x, d.y, d.z);
}

__device__ __forceinline__ bool env_sample(const DScene &S, float u0, float u1, float u2, float u3, f3 &dir,
                                           float &pdf) {
    return env_draw(S.env_prob, S.env_alias, S.env_cpdf, S.env_mw, S.env_mh, u0, u1, u2, u3, dir.x, dir.y, dir.z, pdf);
}

/* Radiance of the environment seen after the first hit (rayPrimary.rmiss.glsl:73-101: HDRI lighting scaled by the
 * intensity for type 1, unscaled for type 2). */
__device__ __forceinline__ f3 env_radiance(const DScene &S, f3 d) {
    const f3 c = env_lookup(S, d);
    return S.env_type == 1u ? S.env_intensity * c : c;
}

/* MIS weight of environment light found by a ray whose direction was sampled with density misp (power heuristic
 * against the environment sample of the extended mode; 1 for camera rays and whenever the environment is not
 * sampled). */
__device__ __forceinline__ float env_mis(const DScene &S, const JobView &J, float misp, f3 d) {
    if (S.env_mw == 0u || J.num_sel == J.num_lights || !(misp >= 0.0f)) return 1.0f;
    return PowerHeuristic(misp, env_pdf_dir(S, normalize(d)) / (float)J.num_sel);
}

/* Cell weights of the importance grid: the largest channel over 4 x 4 points of the cell times sin(theta) of the
 * cell centre. */
__global__ void k_env_importance(DScene S, uint32_t mw, uint32_t mh, float *w) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= mw * mh) return;
    const uint32_t ix = i % mw, iy = i / mw;
    float m = 0.0f;
    for (int sy = 0; sy < 4; ++sy)
        for (int sx = 0; sx < 4; ++sx) {
            const float phi = ((float)ix + (sx + 0.5f) * 0.25f) * (2.0f * PI / (float)mw);
            const float theta = ((float)iy + (sy + 0.5f) * 0.25f) * (PI / (float)mh);
            const f3 c = env_lookup(S, env_dir_of(phi, theta));
            m = fmaxf(m, fmaxf(c.x, fmaxf(c.y, c.z)));
        }
    w[i] = m * sinf(((float)iy + 0.5f) * (PI / (float)mh));
}

/* ------------------------------------------------------- hit geometry -- */
struct Tri3 {
    DVertex v0, v1, v2;
};
/* The vertices of global triangle g (a hit's prim: leaf triangles carry global triangle indices), read from the
 * per-triangle copies, so that neither an index triple nor the instance has to be read first. */
__device__ __forceinline__ void load_tri(const DScene &S, uint32_t g, Tri3 &T) {
    const DVertex *v = S.tri_verts + (size_t)g * 3u;
    T.v0 = v[0];
    T.v1 = v[1];
    T.v2 = v[2];
}
__device__ __forceinline__ void load_rows(const float *src, float *m) {
    const float4 *w = reinterpret_cast<const float4 *>(src);
    const float4 a = w[0], b = w[1], c = w[2];
    m[0] = a.x; m[1] = a.y; m[2] = a.z; m[3] = a.w;
    m[4] = b.x; m[5] = b.y; m[6] = b.z; m[7] = b.w;
    m[8] = c.x; m[9] = c.y; m[10] = c.z; m[11] = c.w;
}

/* process_hit.glsl + construct_frame.glsl */
struct HitGeo {
    f3 wp;
    Frame frame;
    bool flipped;
    float u, v; /* interpolated uvs */
    f3 bary;
};
__device__ __forceinline__ void hit_uv(const Tri3 &T, f3 bary, float &u, float &v) {
    u = T.v0.u * bary.x + T.v1.u * bary.y + T.v2.u * bary.z;
    v = T.v0.v * bary.x + T.v1.v * bary.y + T.v2.v * bary.z;
}
__device__ __forceinline__ void hit_geometry(const DInstance &I, const Tri3 &T, float bu, float bv, f3 rayDir,
                                             HitGeo &g) {
    g.bary = {1.0f - bu - bv, bu, bv};
    hit_uv(T, g.bary, g.u, g.v);
    const f3 b = g.bary;
    const f3 lp = mk(T.v0.px, T.v0.py, T.v0.pz) * b.x + mk(T.v1.px, T.v1.py, T.v1.pz) * b.y +
                  mk(T.v2.px, T.v2.py, T.v2.pz) * b.z;
    float o2w[12], w2o[12];
    load_rows(I.o2w, o2w);
    load_rows(I.w2o, w2o);
    g.wp = xform_point(o2w, lp);
    const f3 ln = mk(T.v0.nx, T.v0.ny, T.v0.nz) * b.x + mk(T.v1.nx, T.v1.ny, T.v1.nz) * b.y +
                  mk(T.v2.nx, T.v2.ny, T.v2.nz) * b.z;
    const f3 lt = mk(T.v0.tx, T.v0.ty, T.v0.tz) * b.x + mk(T.v1.tx, T.v1.ty, T.v1.tz) * b.y +
                  mk(T.v2.tx, T.v2.ty, T.v2.tz) * b.z;
    const f3 lb = mk(T.v0.bx, T.v0.by, T.v0.bz) * b.x + mk(T.v1.bx, T.v1.by, T.v1.bz) * b.y +
                  mk(T.v2.bx, T.v2.by, T.v2.bz) * b.z;
    g.frame.normal = normalize(xform_normal_w2o(w2o, ln));
    g.frame.tangent = normalize(xform_normal_w2o(w2o, lt));
    g.frame.bitangent = normalize(xform_normal_w2o(w2o, lb));
    g.flipped = fixFrame(g.frame.normal, g.frame.tangent, g.frame.bitangent, rayDir);
}

/* Emission with the texture product left out where every emissive slot holds the default white texel (x * 1 = x). */
template <class Fx>
__device__ __forceinline__ f3 mat_emissive_fx(const DScene &S, const DMaterial &m, float tu, float tv) {
    if (!Fx::tex) return m.emissive[3] * mk(m.emissive[0], m.emissive[1], m.emissive[2]);
    return m.emissive[3] * mk(m.emissive[0], m.emissive[1], m.emissive[2]) * tex_rgb(S, m.tex2[0], tu, tv);
}
__device__ __forceinline__ f3 mat_emissive(const DScene &S, const DMaterial &m, float tu, float tv) {
    return m.emissive[3] * mk(m.emissive[0], m.emissive[1], m.emissive[2]) * tex_rgb(S, m.tex2[0], tu, tv);
}
__device__ __forceinline__ float mat_alpha(const DScene &S, const DMaterial &m, float tu, float tv) {
    return m.albedo[3] * tex_sample(S, m.tex2[3], tu, tv).x;
}

/* Volume coefficients (process_volume_hit.glsl:3-8, process_volume_transmittance.glsl:1-10). */
__device__ __forceinline__ f3 vol_sigma_t(const DMaterial &vm) {
    const f3 sa = mk(vm.albedo[0], vm.albedo[1], vm.albedo[2]);
    const f3 ss = vmaxs(mk(vm.mra[0], vm.mra[1], vm.mra[2]), EPSILON);
    return sa + ss;
}
__device__ __forceinline__ f3 vol_transmittance(const DScene &S, uint32_t volIdx, float vtstart, float vtend) {
    const f3 st = vol_sigma_t(S.mats[volIdx]);
    const float dist = fmaxf(vtend - vtstart, EPSILON);
    return vexp(-st * dist);
}

/* ------------------------------------------------------- camera rays -- */
/* raygen.rgen.glsl:63-88 */
__device__ __forceinline__ void camera_ray(const JobView &J, uint32_t px, uint32_t py, Rng &rng, f3 &o, f3 &d) {
    const uint32_t W = J.W, H = J.H;
    const float offx = rnd(rng);
    const float offy = rnd(rng);
    const float uvx = ((float)px + offx) / (float)W;
    const float uvy = ((float)py + offy) / (float)H;
    const float dx = uvx * 2.0f - 1.0f, dy = uvy * 2.0f - 1.0f;
    const float *m = J.pi;
    const float tx = __fmaf_rn(m[0], dx, __fmaf_rn(m[4], dy, m[8] + m[12]));
    const float ty = __fmaf_rn(m[1], dx, __fmaf_rn(m[5], dy, m[9] + m[13]));
    const float tz = __fmaf_rn(m[2], dx, __fmaf_rn(m[6], dy, m[10] + m[14]));
    const float l2 = __fmaf_rn(tx, tx, __fmaf_rn(ty, ty, tz * tz));
    const float inv = 1.0f / sqrtf(l2);
    f3 dc = {tx * inv, ty * inv, tz * inv};
    f3 oc = {0, 0, 0};
    if (J.lens > 0.0f) {
        const float r0 = rnd(rng);
        const float r1 = rnd(rng);
        float lx, ly;
        concentricSampleDisk(r0, r1, lx, ly);
        lx *= J.lens;
        ly *= J.lens;
        const float ft = J.focal / (-dc.z);
        const f3 fp = dc * ft;
        oc = {lx, ly, 0.0f};
        dc = normalize(fp - oc);
    }
    const float *v = J.vi;
    o = {__fmaf_rn(v[0], oc.x, __fmaf_rn(v[4], oc.y, __fmaf_rn(v[8], oc.z, v[12]))),
         __fmaf_rn(v[1], oc.x, __fmaf_rn(v[5], oc.y, __fmaf_rn(v[9], oc.z, v[13]))),
         __fmaf_rn(v[2], oc.x, __fmaf_rn(v[6], oc.y, __fmaf_rn(v[10], oc.z, v[14])))};
    d = {__fmaf_rn(v[0], dc.x, __fmaf_rn(v[4], dc.y, v[8] * dc.z)),
         __fmaf_rn(v[1], dc.x, __fmaf_rn(v[5], dc.y, v[9] * dc.z)),
         __fmaf_rn(v[2], dc.x, __fmaf_rn(v[6], dc.y, v[10] * dc.z))};
}

/* ------------------------------------------------- emitter-lookup helper -- */
/* rayNEE.rahit.glsl:73-131 for an accepted emissive candidate: applies the
 * medium transmittance, rejects back faces and computes the light pdf with the
 * object-space ray origin (gl_ObjectRayOriginEXT).  Returns false if zeroed. */
__device__ __forceinline__ bool nee_emitter(const DScene &S, const JobView &J, const TraceHit &h, f3 origin, f3 dir,
                                            bool inside,
                                            uint32_t volIdx, f3 &T, f3 emissive_in, f3 &e_out, float &pdf_out) {
    const DInstance &I = S.insts[h.inst];
    if (inside) {
        T = T * vol_transmittance(S, volIdx, 0.0001f, h.t);
        if (max3(T) < EPSILON) return false;
    }
    Tri3 Tr;
    load_tri(S, h.prim, Tr);
    const f3 b = {1.0f - h.u - h.v, h.u, h.v};
    float w2o[12], o2w[12];
    load_rows(I.w2o, w2o);
    load_rows(I.o2w, o2w);
    const f3 ln = mk(Tr.v0.nx, Tr.v0.ny, Tr.v0.nz) * b.x + mk(Tr.v1.nx, Tr.v1.ny, Tr.v1.nz) * b.y +
                  mk(Tr.v2.nx, Tr.v2.ny, Tr.v2.nz) * b.z;
    const f3 wn = normalize(xform_normal_w2o(w2o, ln));
    if (dot(wn, dir) > 0.0f) return false; /* back hit */
    const f3 p0 = mk(Tr.v0.px, Tr.v0.py, Tr.v0.pz), p1 = mk(Tr.v1.px, Tr.v1.py, Tr.v1.pz),
             p2 = mk(Tr.v2.px, Tr.v2.py, Tr.v2.pz);
    const f3 wp = xform_point(o2w, p0 * b.x + p1 * b.y + p2 * b.z);
    const f3 w0 = xform_point(o2w, p0), w1 = xform_point(o2w, p1), w2 = xform_point(o2w, p2);
    const float area = 0.5f * length(cross(w1 - w0, w2 - w0));
    const float sampledPointPdf = (1.0f / (float)I.ntri) * (1.0f / area);
    const float dp = dot(-dir, wn);
    if (!(dp > 0.0f)) return false;
    const f3 objOrigin = xform_point(w2o, origin);
    const float lightDirectPdf = sampledPointPdf * distanceSquared(objOrigin, wp) / dp;
    pdf_out = lightDirectPdf * (1.0f / (float)J.num_sel);
    e_out = emissive_in;
    return true;
}

/* Per-candidate material facts used by the any-hit logic. */
struct CandInfo {
    float alpha;
    bool transparent; /* >= 0.99: passes shadow and emitter-lookup rays */
    bool vol_change;
    f3 emissive;
};
template <class Fx = Features<true, true, true, true>>
__device__ __forceinline__ CandInfo cand_info(const DScene &S, const TraceHit &h, bool need_emissive) {
    const DInstance &I = S.insts[h.inst];
    const DMaterial &m = S.inst_mats[h.inst];
    CandInfo c;
    c.transparent = m.mra[3] >= 0.99f;
    c.vol_change = I.idg != I.idb;
    c.emissive = {0, 0, 0};
    c.alpha = 1.0f;
    const bool need_uv = (c.transparent) || (need_emissive && (m.flags & 1u));
    if (need_uv) {
        Tri3 Tr;
        load_tri(S, h.prim, Tr);
        float u, v;
        hit_uv(Tr, mk(1.0f - h.u - h.v, h.u, h.v), u, v);
        const float tu = u * m.tiling[0], tv = v * m.tiling[1];
        if (c.transparent) c.alpha = mat_alpha(S, m, tu, tv);
        if (need_emissive && (m.flags & 1u)) c.emissive = mat_emissive_fx<Fx>(S, m, tu, tv);
    }
    return c;
}

/* Crossing a transparent volume-change surface (raySecondary.rchit.glsl:32-78,
 * rayNEE.rchit.glsl:33-82): new segment origin and volume. */
__device__ __forceinline__ void cross_volume_surface(const DScene &S, const TraceHit &h, f3 dir, bool &inside,
                                                     uint32_t &volIdx, f3 &origin) {
    const DInstance &I = S.insts[h.inst];
    Tri3 Tr;
    load_tri(S, h.prim, Tr);
    HitGeo g;
    hit_geometry(I, Tr, h.u, h.v, dir, g);
    inside = false;
    const float nv = g.flipped ? I.idg : I.idb;
    if (nv != -1.0f) {
        inside = true;
        volIdx = (uint32_t)nv;
    }
    origin = g.wp;
}

/* ------------------------------------------------------------ k_init -- */
template <bool MULTI, class Fx>
__device__ __forceinline__ void start_item(const DScene &S, const RenderParams &P, const PathState &st, uint32_t slot,
                                               uint32_t gitem) {
    uint32_t item = gitem;
    if (MULTI) {
        const uint32_t j = job_of_item(S, gitem);
        st.job[slot] = j;
        item = gitem - S.jobs[j].item_begin;
    }
    const JobView &J = job_of<MULTI>(S, st, slot);
    const uint32_t bl = item / J.npix, pix = item - bl * J.npix;
    const uint32_t px = pix % J.W, py = pix / J.W;
    /* parity: the batch's stream starts here (raygen.rgen.glsl:37); extended: dimension 0 of sample 0 */
    Rng rng = rng_of<Fx>(J, Fx::ext ? 0u : initRNG(px, py, J.W, J.batch_begin + bl, J.seed), item, 0u);
    f3 o, d;
    camera_ray(J, px, py, rng, o, d);
    st.rng[slot] = rng.s;
    if (Fx::nrc && P.nrc) nrc_sample_start(P, J, st, slot, item, 0u);
    st.ctr[slot] = ctr_make(0, 0, 0);
    if (Fx::vol) st.vol[slot] = J.cam_volume >= 0 ? (uint32_t)J.cam_volume : kInvalid;
    st.orig[slot] = st4(o, 0.0f);
    st.dir[slot] = st4(d, 0.0f);
    st.beta[slot] = make_float4(1.f, 1.f, 1.f, -1.f); /* w: last scattering pdf, -1 none */
    st.L[slot] = make_float4(0.f, 0.f, 0.f, 0.f);
    st.accR[slot] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (P.aovs) {
        st.accA[slot] = make_float4(0.f, 0.f, 0.f, 0.f);
        st.accN[slot] = make_float4(0.f, 0.f, 0.f, 0.f);
        st.payA[slot] = make_float4(0.f, 0.f, 0.f, 0.f);
        st.payN[slot] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
}

template <bool MULTI, class Fx>
__global__ __launch_bounds__(kBlock) void k_init(DScene S, RenderParams P, PathState st) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t i0 = i & ~63u;
    uint32_t ishard = shard_of(i0), item = kInvalid;
    const bool need = i < P.nslots;
    item_fetch(P.items, P.items_total, P.items_per_shard, P.item_chunk, need, ishard, item);
    bool active = false;
    if (need) {
        st.item[i] = item;
        st.flags[i] = 0u;
        if (item != kInvalid) {
            start_item<MULTI, Fx>(S, P, st, i, item);
            active = true;
        }
    }
    sq_append(P.ext[0], shard_of(i0), active, i);
}

/* ---------------------------------------------------------- k_extend -- */
template <int STACK, bool COUNT, bool MULTI>
__global__ __launch_bounds__(kTraceBlock) VVPT_TRACE_OCCUPANCY void k_extend(DScene S, RenderParams P, PathState st, uint32_t cur) {
    __shared__ uint2 stack[(STACK + 3) * kTraceBlock]; /* the walk stack + the world ray */
    uint2 *my = stack + threadIdx.x;
    /* the queues that this iteration's k_shade fills; their last consumers ran before this kernel */
    sq_reset(P.ext[cur ^ 1u]);
    sq_reset(P.shd);
    sq_reset(P.sec);
    if (P.nrc_use) sq_reset(P.nrcq);
    const SQueue &Q = P.ext[cur];
    uint32_t nrays = 0;
    TraceCount cnt = {0, 0};
    Trav w;
    bool active = false, done = false, nee = false;
    uint32_t shard = wave_global_id() % kShards, slot = 0;
    for (;;) {
        uint32_t v = 0;
        if (sq_refill(Q, !active, shard, done, v) && !active && !(v & kParked)) {
            slot = v;
            const f3 O = ld3(st.orig[slot]), D = ld3(st.dir[slot]);
            const uint32_t fl = st.flags[slot];
            nee = (fl & F_NEE) != 0u;
            /* with a pending emitter lookup the same walk answers it over [1e-4, ...); a ray that only
             * carries the lookup needs nothing beyond zfar (next_event_estimation.glsl:5) */
            const JobView &J = job_of<MULTI>(S, st, slot);
            trav_init<STACK, kTraceBlock>(w, my, J.tlas_root, O, D, nee ? 0.0001f : 0.001f, 0.001f,
                      (fl & F_TERMINAL) ? fminf(J.zfar, 10000.0f) : 10000.0f, nee ? fminf(J.zfar, 10000.0f) : 0.001f);
            active = true;
            nrays++;
        }
        if (__ballot(active) == 0ull && done) break;
        if (__ballot(active) == 0ull) continue;
        if (active && trav_step<MODE_CLOSEST2, STACK, kTraceBlock, COUNT>(w, S, my, cnt)) {
            const TraceHit &h = w.hit;
            const uint32_t r = 4u * slot;
            st.hit[r] = make_float4(h.t, h.u, h.v, __uint_as_float(h.prim));
            st.hit[r + 1] = make_float4(__uint_as_float(h.inst), __uint_as_float(nee ? w.hitA.inst : 0u),
                                        nee ? w.tskip : 0.0f, 0.0f);
            if (nee) {
                st.hit[r + 2] = make_float4(w.hitA.t, w.hitA.u, w.hitA.v, __uint_as_float(w.hitA.prim));
                st.hit[r + 3] = make_float4(0.0f, 0.0f, 0.0f, 0.0f); /* the whole line, no partial sector */
            }
            active = false;
        }
    }
    wave_add64(P.stats, S_PATH, nrays);
    if (COUNT) {
        wave_add64(P.stats, S_NODES_EXT, cnt.nodes);
        wave_add64(P.stats, S_TRIS_EXT, cnt.tris);
    }
}

/* ---------------------------------------------------------- k_shade -- */
struct ShadeOut {
    uint32_t secmask;
};

/* lightSampling.glsl:1-106 without the shadow loop: returns the light sample,
 * radiance before visibility, and the segment length for the shadow ray. */
struct LightSample {
    f3 dir, radiance;
    float pdf, tmax;
    bool delta;
};
template <class Fx>
__device__ __forceinline__ LightSample sample_light(const DScene &S, const JobView &J, Rng &rng, f3 P, bool env_last) {
    LightSample ls;
    ls.delta = true;
    ls.radiance = {0, 0, 0};
    ls.pdf = 1.0f;
    ls.dir = {0, 0, 0};
    ls.tmax = 10000.0f;
    const uint32_t total = J.num_sel; /* num_lights, plus the environment in the extended mode */
    if (total == 0u) return ls;
    const float pdf = 1.0f / (float)total;
    const uint32_t li = min((uint32_t)(rnd(rng) * (float)total), total - 1u);
    if (Fx::ext && li >= J.num_lights) {
        /* extended mode: an environment sample, shadowed like a directional light */
        const float u0 = rnd(rng), u1 = rnd(rng), u2 = rnd(rng), u3 = rnd(rng);
        f3 dir;
        float ep;
        if (!env_last && env_sample(S, u0, u1, u2, u3, dir, ep)) {
            ls.dir = dir;
            ls.radiance = env_radiance(S, dir);
            ls.pdf = ep * pdf;
            ls.delta = false;
            ls.tmax = fminf((float)(uint32_t)J.zfar, 10000.0f);
        }
        return ls;
    }
    const DLight L = S.lights[J.light_begin + li];
    const f3 col = mk(L.color[0], L.color[1], L.color[2]);
    const f3 pos = mk(L.position[0], L.position[1], L.position[2]);
    if (L.type == 0u) {
        const f3 dv = pos - P;
        ls.tmax = length(dv);
        ls.dir = dv / ls.tmax;
        const float dd = length(P - pos);
        ls.radiance = col * (1.0f / (dd * dd)) * L.intensity;
        ls.pdf = pdf;
    } else if (L.type == 1u) {
        ls.dir = -pos;
        ls.tmax = J.zfar;
        ls.radiance = col * L.intensity;
        ls.pdf = pdf;
    } else {
        const DInstance &I = S.insts[L.inst];
        const DMaterial &m = S.inst_mats[L.inst];
        const uint32_t tri = (uint32_t)(rnd(rng) * (float)I.ntri);
        const float trianglePdf = 1.0f / (float)I.ntri;
        const float r0 = rnd(rng);
        const float r1 = rnd(rng);
        const float a = sqrtf(1.0f - r0);
        const f3 sb = {1.0f - a, a * r1, 1.0f - (1.0f - a) - a * r1};
        Tri3 Tr;
        load_tri(S, I.idx_offset + tri, Tr);
        float o2w[12], w2o[12];
        load_rows(I.o2w, o2w);
        load_rows(I.w2o, w2o);
        const f3 p0 = mk(Tr.v0.px, Tr.v0.py, Tr.v0.pz), p1 = mk(Tr.v1.px, Tr.v1.py, Tr.v1.pz),
                 p2 = mk(Tr.v2.px, Tr.v2.py, Tr.v2.pz);
        const f3 q0 = xform_point(o2w, p0), q1 = xform_point(o2w, p1), q2 = xform_point(o2w, p2);
        const float area = 0.5f * length(cross(q1 - q0, q2 - q0));
        const float sampledPointPdf = 1.0f / area;
        f3 sp = p0 * sb.x + p1 * sb.y + p2 * sb.z;
        f3 sn = mk(Tr.v0.nx, Tr.v0.ny, Tr.v0.nz) * sb.x + mk(Tr.v1.nx, Tr.v1.ny, Tr.v1.nz) * sb.y +
                mk(Tr.v2.nx, Tr.v2.ny, Tr.v2.nz) * sb.z;
        const float su = Tr.v0.u * sb.x + Tr.v1.u * sb.y + Tr.v2.u * sb.z;
        const float sv = Tr.v0.v * sb.x + Tr.v1.v * sb.y + Tr.v2.v * sb.z;
        sp = xform_point(o2w, sp);
        sn = xform_normal_w2o(w2o, sn);
        const f3 dv = sp - P;
        ls.tmax = length(dv);
        ls.dir = dv / ls.tmax;
        const float dp = dot(-ls.dir, sn);
        if (dp > 0.0f) {
            ls.radiance = mat_emissive_fx<Fx>(S, m, su * m.tiling[0], sv * m.tiling[1]);
            ls.pdf = pdf * trianglePdf * sampledPointPdf * distanceSquared(P, sp) / dp;
        } else {
            ls.radiance = {0, 0, 0};
            ls.pdf = 0.0f;
        }
        ls.delta = false;
    }
    return ls;
}

/* Storage index of secondary record r = 3 slot + k. */
__device__ __forceinline__ uint32_t sec_ix(const PathState &st, uint32_t r) { return (r % 3u) * st.nsec + r / 3u; }

__device__ __forceinline__ void emit_sec(const RenderParams &P, const PathState &st, uint32_t slot, uint32_t k, f3 o,
                                         float w_o, f3 d, float w_d, f3 c, uint32_t vol) {
    const uint32_t r = k * st.nsec + slot;
    st.sec_o[r] = st4(o, w_o);
    st.sec_d[r] = st4(d, w_d);
    st.sec_c[r] = st4(c, 0.0f);
    if (P.media) st.sec_v[r] = vol;
}

/* process_volume_hit.glsl:1-45 (sampling part).  Returns sampledMedium, updates beta. */
__device__ __forceinline__ bool volume_sample(const DScene &S, uint32_t volIdx, Rng &rng, f3 &beta, float vtstart,
                                              float vtend, float &hit_distance, float &g) {
    const DMaterial vm = S.mats[volIdx];
    const f3 sigma_s = vmaxs(mk(vm.mra[0], vm.mra[1], vm.mra[2]), EPSILON);
    const f3 sigma_t = mk(vm.albedo[0], vm.albedo[1], vm.albedo[2]) + sigma_s;
    g = fmaxf(fminf(vm.emissive[0], 0.99f), -0.99f);
    const float dist_in = fmaxf(vtend - vtstart, EPSILON);
    const uint32_t channel = min((uint32_t)(rnd(rng) * 3.0f), 2u);
    const float st_c = channel == 0u ? sigma_t.x : (channel == 1u ? sigma_t.y : sigma_t.z);
    hit_distance = -logf(1.0f - rnd(rng)) / st_c;
    const bool sampled = hit_distance < dist_in;
    const float td = fminf(hit_distance, dist_in);
    const f3 tr = vexp(-sigma_t * td);
    const f3 density = sampled ? (sigma_t * tr) : tr;
    float pdf = 0.0f;
    pdf += density.x;
    pdf += density.y;
    pdf += density.z;
    pdf *= 0.3333333f;
    if (pdf == 0.0f) pdf = 1.0f;
    const f3 F = sampled ? (tr * sigma_s / pdf) : (tr / pdf);
    beta = beta * F;
    return sampled;
}

/* One bounce of slot `slot`, whose flags word is flags_in and whose radiance so far is L.  Returns the mask of
 * secondary records it wrote (and F_NRCQ, F_NRC_FALLBACK); `over` is set when the sample has ended.  A sample that
 * ends with nothing pending leaves no state behind but its radiance in L and its generator state in rng_out. */
template <class Fx>
__device__ __forceinline__ uint32_t shade_one(const DScene &S, const JobView &J, const RenderParams &P, const PathState &st,
                                              uint32_t slot, uint32_t flags_in, uint32_t ctr, f3 &L, uint32_t &rng_out,
                                              bool &over) {
    {
        uint32_t flags = flags_in & F_NEE;
        Rng rng = rng_of<Fx>(J, st.rng[slot], Fx::ext ? st.item[slot] - J.item_begin : 0u, ctr_sample(ctr));
        const uint32_t d = ctr_depth(ctr);
        uint32_t sdepth = ctr_sdepth(ctr);
        uint32_t vol = kInvalid;
        if (Fx::vol) vol = st.vol[slot];
        bool inside = Fx::vol && vol != kInvalid;
        const float4 beta4 = st.beta[slot];
        f3 beta = ld3(beta4);
        /* extended mode: pdf of the direction sampled at the last scattering vertex (-1: a camera ray), the BSDF
         * side of the MIS pair for environment light found by this ray */
        float misp = beta4.w;
        const bool env_last = d + 1u >= J.depth; /* no environment sample where the BSDF side cannot follow */
        const f3 O = ld3(st.orig[slot]);
        const f3 D = ld3(st.dir[slot]);
        uint32_t secmask = 0;

        /* (1) emitter lookup of the previous bounce (next_event_estimation.glsl) */
        if (flags & F_NEE) {
            const float4 ha = st.hit[4u * slot + 2u], hi = st.hit[4u * slot + 1u];
            TraceHit hA = {ha.x, ha.y, ha.z, __float_as_uint(hi.y), __float_as_uint(ha.w)};
            const float4 nb = st.nee[slot];
            /* hA is the first candidate that is not passed (INST_NEE_PASS instances are transparent,
             * non-emissive and keep the volume: rayNEE.rahit.glsl:43-70 only scales their throughput) */
            if (hA.prim != kInvalid && hA.t <= J.zfar) {
                const CandInfo c = cand_info<Fx>(S, hA, true);
                if (isBlackEps(c.emissive, 0.05f)) {
                    if (c.transparent) {
                        /* a transparent surface that changes volume (or whose emission texture is black
                         * here): the general closest-first walk */
                        emit_sec(P, st, slot, 1, O, 0.0f, D, nb.w, ld3(nb), vol);
                        secmask |= F_SEC1;
                    }
                } else {
                    f3 T = {1, 1, 1}, e;
                    float lpdf = 0.0f;
                    if (nee_emitter(S, J, hA, O, D, inside, vol, T, c.emissive, e, lpdf)) {
                        const float w = PowerHeuristic(nb.w, lpdf);
                        const f3 contrib = w * T * e * ld3(nb);
                        if (hi.z < hA.t) {
                            /* passed surfaces in front of the emitter: their 1 - alpha product */
                            emit_sec(P, st, slot, 1, O, __uint_as_float(__float_as_uint(hA.t) - 1u), D, 0.0f, contrib,
                                     kInvalid);
                            secmask |= F_SEC1 | F_TPASS;
                        } else {
                            L = L + contrib;
                        }
                    }
                }
            }
            flags &= ~F_NEE;
        }
        if (flags_in & F_TERMINAL) {
            /* the walk only answered the last bounce's emitter lookup: the sample is over */
            rng_out = rng.s;
            over = true;
            return secmask;
        }

        /* (2) the path bounce */
        const float4 hb = st.hit[4u * slot], hbi = st.hit[4u * slot + 1u];
        const TraceHit h = {hb.x, hb.y, hb.z, __float_as_uint(hbi.x), __float_as_uint(hb.w)};
        bool stop = false, nee_pending = false, do_rr = true;
        f3 nO = O, nD = D;
        float neePdf = 0.0f;
        f3 neeBeta = {0, 0, 0};
        bool sampledMedium = false;
        float vhd = 0.0f, g = 0.0f;
        if (Fx::vol && inside) {
            const float vtend = h.prim != kInvalid ? h.t : fminf((float)(uint32_t)J.zfar, 10000.0f);
            sampledMedium = volume_sample(S, vol, rng, beta, 0.001f, vtend, vhd, g);
        }
        if (Fx::vol && sampledMedium) {
            /* process_volume_hit.glsl:42-79: scattering event */
            const f3 wrd = normalize(D);
            const f3 wo = -wrd;
            const f3 sp = O + (0.001f + vhd) * wrd;
            const LightSample ls = sample_light<Fx>(S, J, rng, sp, env_last);
            if (!isBlack(ls.radiance)) {
                const float p = HenyeyGreenstein(dot(wo, ls.dir), g);
                if (p != 0.0f) {
                    const f3 F = {p, p, p};
                    f3 c;
                    if (ls.delta)
                        c = ls.radiance * F * beta / ls.pdf;
                    else
                        c = PowerHeuristic(ls.pdf, p) * ls.radiance * F * beta / ls.pdf;
                    emit_sec(P, st, slot, 0, sp, ls.tmax, ls.dir, 0.0f, c, vol);
                    secmask |= F_SEC0;
                }
            }
            f3 wi;
            const float r0 = rnd(rng);
            const float r1 = rnd(rng);
            neePdf = HG_Sample(wo, wi, r0, r1, g);
            nO = sp;
            nD = wi;
            nee_pending = true;
            neeBeta = beta;
            misp = neePdf;
        } else if (h.prim == kInvalid) {
            /* rayPrimary.rmiss.glsl:53-103 */
            stop = true;
            do_rr = false;
            const f3 bg = mk(S.bg[0], S.bg[1], S.bg[2]);
            /* the environment's radiance along the ray: the background colour (type 0, and camera rays of type 2), the
             * map (scaled by the intensity for type 1) */
            f3 c = bg;
            const bool map = S.env_type == 1u || (S.env_type == 2u && sdepth != 0u);
            if (map) {
                c = env_lookup(S, D);
                if (S.env_type == 1u) c = S.env_intensity * c;
            }
            if (S.env_type <= 2u) {
                if (P.aovs && sdepth == 0u) {
                    st.payA[slot] = st4(c, 0.f);
                    st.payN[slot] = make_float4(0.f, 0.f, 0.f, 0.f);
                }
                if (Fx::ext && map)
                    L = L + env_mis(S, J, misp, D) * c * beta;
                else
                    L = L + c * beta;
            }
        } else {
            /* rayPrimary{Lambert,PBRStandard}.rchit.glsl:60-172 */
            const DInstance &I = S.insts[h.inst];
            const DMaterial m = S.inst_mats[h.inst];
            Tri3 Tr;
            load_tri(S, h.prim, Tr);
            HitGeo gg;
            hit_geometry(I, Tr, h.u, h.v, D, gg);
            const float tu = gg.u * m.tiling[0], tv = gg.v * m.tiling[1];
            const bool isPBR = m.tiling[2] == 0.0f;
            bool passed = false;
            if (m.mra[3] > 0.0f) {
                const float alpha = mat_alpha(S, m, tu, tv);
                const float ra = rnd(rng);
                if (alpha < EPSILON || ra > alpha) {
                    if (Fx::vol && I.idg != I.idb) {
                        inside = false;
                        const float nv = gg.flipped ? I.idg : I.idb;
                        if (nv != -1.0f) {
                            inside = true;
                            vol = (uint32_t)nv;
                        }
                        if (!inside) vol = kInvalid;
                    }
                    nO = gg.wp;
                    nD = normalize(D);
                    passed = true;
                    do_rr = false;
                }
            }
            if (!passed) {
                Frame fr = gg.frame;
                /* without textures every slot holds its default texel: white (x * 1 = x) or the flat normal */
                applyNormalToFrame(fr, processNormalFromNormalMap(
                                           Fx::tex ? tex_rgb(S, m.tex2[1], tu, tv)
                                                   : mk(S.flat_normal[0], S.flat_normal[1], S.flat_normal[2])));
                f3 albedo = mk(m.albedo[0], m.albedo[1], m.albedo[2]);
                if (Fx::tex) albedo = albedo * tex_rgb(S, m.tex1[0], tu, tv);
                PBRStd pbr;
                if (isPBR) {
                    pbr.albedo = albedo;
                    pbr.metallic = Fx::tex ? m.mra[0] * tex_sample(S, m.tex1[1], tu, tv).x : m.mra[0];
                    pbr.roughness = fmaxf(Fx::tex ? m.mra[1] * tex_sample(S, m.tex1[2], tu, tv).x : m.mra[1], 0.035f);
                }
                const f3 emissive = (m.flags & 1u) ? mat_emissive_fx<Fx>(S, m, tu, tv) : mk(0, 0, 0);
                if (sdepth == 0u && P.aovs) {
                    st.payA[slot] = st4(albedo, 0.f);
                    st.payN[slot] = st4(fr.normal * 0.5f + mk(0.5f, 0.5f, 0.5f), 0.f);
                }
                if (sdepth == 0u && !isBlackEps(emissive, isPBR ? 0.1f : 0.05f) && !gg.flipped) {
                    L = L + emissive * beta;
                    stop = true;
                    do_rr = false;
                } else {
                    sdepth += 1u;
                    bool cached = false;
                    if (Fx::nrc && P.nrc) {
                        /* path spread (Müller et al. 2021): footprint a0 = d^2 / (4 pi cos) at the primary vertex,
                         * then sum of sqrt(d^2 / (p cos)) over the vertices after it */
                        const float cosn = fmaxf(fabsf(dot(fr.normal, D)), 1e-4f);
                        float2 sp = st.spread[slot];
                        if (sdepth == 1u)
                            sp = make_float2(h.t * h.t / (4.0f * PI * cosn), 0.0f);
                        else
                            sp.y += sqrtf(h.t * h.t / (fmaxf(misp, 1e-8f) * cosn));
                        st.spread[slot] = sp;
                        const float rough = isPBR ? pbr.roughness : 1.0f;
                        const uint32_t tw = st.nrct[slot];
                        if (tw != kInvalid) {
                            /* training sample: record the vertex (input, radiance so far, throughput); the low 24
                             * bits of nrct name the sample's record block, the top 8 count its records */
                            const uint32_t tb = tw & 0x00ffffffu;
                            if (sdepth <= P.nrc_vmax) {
                                st.nrct[slot] = tb | (sdepth << 24);
                                float4 *r = reinterpret_cast<float4 *>(P.nrc_pool +
                                                                       ((size_t)tb * P.nrc_vmax + sdepth - 1u) * 16u);
                                r[0] = make_float4(gg.wp.x, gg.wp.y, gg.wp.z, -D.x);
                                r[1] = make_float4(-D.y, -D.z, rough, albedo.x);
                                r[2] = make_float4(albedo.y, albedo.z, L.x, L.y);
                                r[3] = make_float4(L.z, beta.x, beta.y, beta.z);
                            }
                        } else if (P.nrc_use && sdepth > 1u && sp.y * sp.y > P.nrc_c * sp.x &&
                                   !nrc_region_ok(P, gg.wp)) {
                            secmask |= F_NRC_FALLBACK;
                        } else if (P.nrc_use && sdepth > 1u && sp.y * sp.y > P.nrc_c * sp.x) {
                            /* the rest of the path comes from the cache: inputs for the query */
                            st.orig[slot] = make_float4(gg.wp.x, gg.wp.y, gg.wp.z, rough);
                            st.dir[slot] = make_float4(-D.x, -D.y, -D.z, 0.0f);
                            st.nee[slot] = st4(albedo, 0.0f);
                            cached = true;
                            stop = true;
                            do_rr = false;
                            secmask |= F_NRCQ;
                        }
                    }
                    f3 wo = worldToLocal(fr, -D);
                    {
                        /* the cosine with its rounding fixed (the last product is rounded before it is added), so that
                         * every Features variant makes the same image whatever else the compiler can share it with */
#pragma clang fp contract(off)
                        const float xy = __fmaf_rn(D.y, fr.normal.y, D.x * fr.normal.x);
                        wo.y = -(xy + D.z * fr.normal.z);
                    }
                    const LightSample ls = cached ? LightSample{{0, 0, 0}, {0, 0, 0}, 1.0f, 0.0f, true}
                                                  : sample_light<Fx>(S, J, rng, gg.wp, env_last);
                    if (!isBlack(ls.radiance)) {
                        const f3 wi = worldToLocal(fr, ls.dir);
                        f3 F;
                        if (isPBR)
                            F = evalPBRStandard(pbr, wi, wo, normalize(wo + wi));
                        else
                            F = albedo * INV_PI * clampf(wi.y, 0.0f, 1.0f);
                        if (!isBlack(F)) {
                            f3 c;
                            if (ls.delta) {
                                c = ls.radiance * F * beta / ls.pdf;
                            } else {
                                const float bp = isPBR ? pdfPBRStandard(wi, wo, pbr)
                                                       : cosineSampleHemispherePdf(clampf(wi.y, 0.0f, 1.0f));
                                c = PowerHeuristic(ls.pdf, bp) * ls.radiance * F * beta / ls.pdf;
                            }
                            emit_sec(P, st, slot, 0, gg.wp, ls.tmax, ls.dir, 0.0f, c, vol);
                            secmask |= F_SEC0;
                        }
                    }
                    float sdp = 0.0f;
                    if (cached) {
                    } else if (isPBR) {
                        const float u0 = rnd(rng);
                        const float u1 = rnd(rng);
                        const float u2 = rnd(rng);
                        f3 sdl;
                        const f3 F = samplePBRStandard(sdl, wo, sdp, pbr, u0, u1, u2);
                        nO = gg.wp;
                        nD = localToWorld(fr, sdl);
                        if (isBlack(F)) {
                            stop = true;
                            do_rr = false;
                        } else {
                            const f3 r = F / sdp;
                            beta = beta * mk(clampf(r.x, 0.f, 1.f), clampf(r.y, 0.f, 1.f), clampf(r.z, 0.f, 1.f));
                        }
                    } else {
                        const float u0 = rnd(rng);
                        const float u1 = rnd(rng);
                        const f3 sdl = cosineSampleHemisphere(u0, u1, sdp);
                        nO = gg.wp;
                        nD = localToWorld(fr, sdl);
                        beta = beta * albedo;
                    }
                    if (!stop) {
                        nee_pending = true;
                        neePdf = sdp;
                        neeBeta = beta;
                        misp = sdp;
                    }
                }
            }
        }
        /* russian_roulette.glsl:1-11 */
        if (do_rr && !stop) {
            const float rr = rnd(rng);
            if (d > RUSSIAN_ROULETTE_DEPTH) {
                const float maxBeta = fmaxf(beta.x, fmaxf(beta.y, beta.z));
                if (rr >= maxBeta)
                    stop = true;
                else
                    beta = beta * (1.0f / maxBeta);
            }
        }
        const bool cont = !stop && (d + 1u < J.depth);
        if (cont) {
            st.orig[slot] = st4(nO, 0.f);
            st.dir[slot] = st4(nD, 0.f);
            st.ctr[slot] = ctr_make(ctr_sample(ctr), d + 1u, sdepth);
            if (nee_pending) {
                flags |= F_NEE;
                st.nee[slot] = st4(neeBeta, neePdf);
            }
        } else if (nee_pending) {
            /* The path ends (Russian roulette or depth) but its emitter lookup along the sampled direction
             * is still owed (next_event_estimation.glsl runs before russian_roulette.glsl): it rides on one
             * more extension walk over [1e-4, zfar] and is resolved by the next k_shade. */
            st.orig[slot] = st4(nO, 0.f);
            st.dir[slot] = st4(nD, 0.f);
            st.nee[slot] = st4(neeBeta, neePdf);
            flags |= F_NEE | F_TERMINAL;
        } else {
            over = true;
            rng_out = rng.s;
            if (secmask & F_NRCQ) st.beta[slot] = st4(beta, misp); /* the query's weight */
            return secmask;
        }
        st.beta[slot] = st4(beta, misp);
        st.L[slot] = st4(L, 0.f);
        st.rng[slot] = rng.s;
        if (Fx::vol) st.vol[slot] = inside ? vol : kInvalid;
        st.flags[slot] = flags | (secmask & ~F_NRC_FALLBACK);
        return secmask;
    }
}

/* Completion bookkeeping of a batched render: the lanes of a wave that ended a work item subtract their count from
 * their job's remaining items with one atomic per job present in the wave (same-address atomics serialize in L2,
 * and every item of a large job would otherwise hit the one counter); the lane that takes a counter to zero stamps
 * the job's completion time.  Called in wave-uniform control flow; `job` is kInvalid for lanes that ended nothing. */
__device__ __forceinline__ void job_items_done(const DScene &S, uint32_t job) {
    unsigned long long m = __ballot(job != kInvalid);
    const uint32_t lane = __lane_id();
    while (m != 0ull) {
        const int leader = __ffsll((long long)m) - 1;
        const uint32_t lj = __shfl(job, leader);
        const unsigned long long same = __ballot(job == lj);
        if ((int)lane == leader) {
            const uint32_t n = (uint32_t)__popcll(same);
            const JobView &J = S.jobs[lj];
            if (atomicSub(J.remaining, n) == n) *J.done_ticks = wall_clock64();
        }
        m &= ~same;
    }
}

/* Arguments of k_shade, read where they are used: a by-value kernel argument is loaded whole at the kernel's entry and
 * held in scalar registers to its end, and these 900 bytes spilled 229 of them (2,600 v_readlane in the code).  The
 * empty asm keeps the loads behind this point; they are scalar loads from the constant kernel-argument segment. */
struct ShadeArgs {
    DScene S;
    RenderParams P;
    PathState st;
    uint32_t cur;
};
template <class T>
__device__ __forceinline__ const T &kernargs() {
    const __attribute__((address_space(4))) char *p =
        (const __attribute__((address_space(4))) char *)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const T *)(const char *)p;
}

/* Second half of k_shade for one wave's slots (shard sh, every lane calls it): ends the samples that are over
 * (raygen.rgen.glsl:126-128), refills ended work items and appends the slots that go on to the next queue. */
template <bool MULTI, class Fx>
__device__ __forceinline__ void end_samples(uint32_t nxt, uint32_t sh, bool valid, bool over, bool parked, uint32_t slot,
                                            uint32_t ctr, uint32_t rng_s, f3 L) {
    const ShadeArgs &A = kernargs<ShadeArgs>();
    const DScene &S = A.S;
    const RenderParams &P = A.P;
    const PathState &st = A.st;
    uint32_t s = 0, ended_job = kInvalid;
    bool item_end = false, push = valid && !over;
    f3 accR = {0, 0, 0}, accA = {0, 0, 0}, accN = {0, 0, 0};
    if (over) {
        if (Fx::nrc && P.nrc) {
            const uint32_t tw = st.nrct[slot];
            if (tw != kInvalid) nrc_emit_training(P, tw & 0x00ffffffu, tw >> 24, L);
        }
        const JobView &J = job_of<MULTI>(S, st, slot);
        accR = ld3(st.accR[slot]) + L / J.total_samples;
        s = ctr_sample(ctr) + 1u;
        if (P.aovs) {
            accA = ld3(st.accA[slot]) + ld3(st.payA[slot]) / J.total_samples;
            accN = ld3(st.accN[slot]) + ld3(st.payN[slot]) / J.total_samples;
        }
        item_end = s == J.batch_size;
    }
    /* finished work items take new ones from the wave's item shard */
    uint32_t ishard = sh, newitem = kInvalid;
    item_fetch(P.items, P.items_total, P.items_per_shard, P.item_chunk, item_end, ishard, newitem);
    if (over) {
        const uint32_t item = st.item[slot];
        if (item_end) {
            P.partR[item] = st4(accR, 0.f);
            if (P.aovs) {
                P.partA[item] = st4(accA, 0.f);
                P.partN[item] = st4(accN, 0.f);
            }
            if (MULTI) ended_job = st.job[slot]; /* counted below, once per job and wave */
            st.item[slot] = newitem;
            if (newitem != kInvalid) {
                start_item<MULTI, Fx>(S, P, st, slot, newitem);
                push = true;
            }
        } else {
            const JobView &J = job_of<MULTI>(S, st, slot);
            const uint32_t litem = item - J.item_begin;
            const uint32_t pix = litem % J.npix;
            /* parity: the batch's stream continues; extended: dimension 0 of the next sample */
            Rng rng = rng_of<Fx>(J, Fx::ext ? 0u : rng_s, litem, s);
            f3 o, d;
            camera_ray(J, pix % J.W, pix / J.W, rng, o, d);
            if (Fx::nrc && P.nrc) nrc_sample_start(P, J, st, slot, litem, s);
            st.orig[slot] = st4(o, 0.f);
            st.dir[slot] = st4(d, 0.f);
            st.beta[slot] = make_float4(1.f, 1.f, 1.f, -1.f); /* w: last scattering pdf, -1 none */
            st.L[slot] = make_float4(0.f, 0.f, 0.f, 0.f);
            st.ctr[slot] = ctr_make(s, 0, 0);
            if (Fx::vol) st.vol[slot] = J.cam_volume >= 0 ? (uint32_t)J.cam_volume : kInvalid;
            st.rng[slot] = rng.s;
            st.accR[slot] = st4(accR, 0.f);
            if (P.aovs) {
                st.accA[slot] = st4(accA, 0.f);
                st.accN[slot] = st4(accN, 0.f);
            }
            push = true;
        }
        st.flags[slot] = 0u;
    }
    if (MULTI) job_items_done(S, ended_job);
    sq_append(P.ext[nxt], sh, push, parked ? slot | kParked : slot);
}

/* k_shade: one pass over the extension queue's slots: results of the previous bounce's secondary records are added,
 * the bounce is shaded, and a sample that is over with nothing pending ends here - its radiance goes to the slot's
 * accumulators, finished work items are written and replaced, the next camera ray is made - before the wave appends
 * its slots to the next extension queue.  A sample that is over but waits for records of its last bounce or for a
 * cache query is parked: its queue entry carries kParked and the next pass ends it.
 *
 * Bound by its dependent gathers (path state, hit, instance, triangle, light).  It takes 145 to 168 VGPRs, 3 waves per
 * SIMD, without scratch memory; every variant is held to that.  At 4 waves (128 VGPRs, up to 32 bytes of scratch per
 * lane) the benchmark's 1080p field took 138.6 instead of 140.0 ms a frame, but both GPU memory faults this kernel's
 * builds have seen came with variants that spilled, and their cause is not shown.
 * One pass instead of two (a kernel of its own to end samples read the queue, flags and radiance again and wrote them
 * again), code for the scene's features only (textures that are the default texel cost two dependent loads each) and
 * arguments read in place took the 1080p field at 64 spp from 150 to 136 ms, the 1080p medium at 32
 * spp from 202 to 180 ms and a 64x64 preview from 3.2 to 3.0 ms. */
template <bool MULTI, class Fx>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(3, 8))) void k_shade(ShadeArgs) {
    __shared__ SQView view;
    const ShadeArgs &A0 = kernargs<ShadeArgs>();
    const uint32_t cur = A0.cur;
    const uint32_t nxt = cur ^ 1u;
    sq_view_load(A0.P.ext[cur], view);
    const uint32_t count = view.pre[kShards];
    const uint32_t stride = gridDim.x * blockDim.x;
    for (uint32_t base = blockIdx.x * blockDim.x; base < count; base += stride) {
        const ShadeArgs &A = kernargs<ShadeArgs>();
        const DScene &S = A.S;
        const RenderParams &P = A.P;
        const PathState &st = A.st;
        const uint32_t i = base + threadIdx.x;
        const uint32_t sh = shard_of(i & ~63u);
        const bool valid = i < count;
        uint32_t slot = 0, secmask = 0, ctr = 0, rng_s = 0;
        f3 L = {0, 0, 0};
        bool simple = true, over = false, parked = false;
        if (valid) {
            slot = sq_at(P.ext[cur], view, i) & ~kParked;
            const JobView &J = job_of<MULTI>(S, st, slot);
            simple = !(J.scene_flags & SCENE_HAS_VOLUME_CHANGE);
            const uint32_t flags = st.flags[slot];
            ctr = st.ctr[slot];
            L = ld3(st.L[slot]);
            if (flags & F_SEC0) L = L + ld3(st.sec_c[slot]);
            if (flags & F_SEC1) L = L + ld3(st.sec_c[st.nsec + slot]);
            if (flags & F_SEC2) L = L + ld3(st.sec_c[2u * st.nsec + slot]);
            if (flags & F_DONE) {
                over = true;
                rng_s = st.rng[slot];
            } else {
                secmask = shade_one<Fx>(S, J, P, st, slot, flags, ctr, L, rng_s, over);
                if (over && (secmask & (F_SEC0 | F_SEC1 | F_SEC2 | F_NRCQ))) {
                    over = false;
                    parked = true;
                    st.L[slot] = st4(L, 0.f);
                    st.rng[slot] = rng_s;
                    st.flags[slot] = F_DONE | (secmask & (F_SEC0 | F_SEC1 | F_SEC2 | F_TPASS));
                }
            }
        }
        /* single-segment shadow rays and 1 - alpha products go to the persistent shadow walk, the rest to the
         * general walk */
        const bool to_shd = simple && (secmask & F_SEC0);
        const bool tpass = (secmask & F_TPASS) != 0u;
        uint32_t gen = to_shd ? (secmask & ~F_SEC0) : secmask;
        if (tpass) gen &= ~F_SEC1;
        sq_append(P.shd, sh, to_shd, slot * 3u);
        sq_append(P.shd, sh, tpass, slot * 3u + 1u);
        sq_append(P.sec, sh, (gen & F_SEC0) != 0u, slot * 3u + 0u);
        sq_append(P.sec, sh, (gen & F_SEC1) != 0u, slot * 3u + 1u);
        sq_append(P.sec, sh, (gen & F_SEC2) != 0u, slot * 3u + 2u);
        if (Fx::nrc && P.nrc_use) {
            sq_append(P.nrcq, sh, (secmask & F_NRCQ) != 0u, slot);
            wave_add64(P.stats, S_NRC_FALLBACK, (secmask & F_NRC_FALLBACK) ? 1u : 0u);
        }
        end_samples<MULTI, Fx>(nxt, sh, valid, over, parked, slot, ctr, rng_s, L);
    }
}

/* ------------------------------------------------------ cache queries -- */
/* Gathers the inputs of this iteration's cache queries into a dense batch (count to nrc_ctr[2]). */
__global__ __launch_bounds__(kBlock) void k_nrc_gather(RenderParams P, PathState st) {
    __shared__ SQView view;
    sq_view_load(P.nrcq, view);
    const uint32_t count = view.pre[kShards];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        P.nrc_ctr[2] = count;
        atomicAdd(&P.stats[S_NRCQ], (unsigned long long)count);
    }
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x) {
        const uint32_t slot = sq_at(P.nrcq, view, i);
        const float4 o = st.orig[slot], d = st.dir[slot], a = st.nee[slot];
        float *q = P.nrc_qin + (size_t)i * 10u;
        q[0] = o.x; q[1] = o.y; q[2] = o.z;
        q[3] = d.x; q[4] = d.y; q[5] = d.z;
        q[6] = o.w;
        q[7] = a.x; q[8] = a.y; q[9] = a.z;
        P.nrc_qslot[i] = slot;
    }
}

/* Adds throughput x cached radiance to each querying path (clamped at zero). */
__global__ __launch_bounds__(kBlock) void k_nrc_apply(RenderParams P, PathState st) {
    const uint32_t count = P.nrc_ctr[2];
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x) {
        const uint32_t slot = P.nrc_qslot[i];
        const f3 b = ld3(st.beta[slot]);
        const float *y = P.nrc_qpred + (size_t)i * 3u;
        const f3 c = mk(fmaxf(y[0], 0.0f), fmaxf(y[1], 0.0f), fmaxf(y[2], 0.0f));
        st.L[slot] = st4(ld3(st.L[slot]) + b * c, 0.0f);
    }
}

/* ------------------------------------------------------- k_secondary -- */
/* Any-hit callback of shadow rays in scenes without volume-changing surfaces
 * (raySecondary.rahit.glsl:31-72): returns true to stop the walk. */
struct ShadowAnyHit {
    const DScene *S;
    float T;
    bool shadowed;
    bool eps_rule; /* shadow rays stop at T <= EPSILON; 1 - alpha products for emitter lookups do not */
    __device__ __forceinline__ bool operator()(const TraceHit &h) {
        const DInstance &I = S->insts[h.inst];
        if (!(I.flags & INST_TRANSPARENT)) {
            shadowed = true;
            return true;
        }
        const DMaterial &m = S->inst_mats[h.inst];
        Tri3 Tr;
        load_tri(*S, h.prim, Tr);
        float u, v;
        hit_uv(Tr, mk(1.0f - h.u - h.v, h.u, h.v), u, v);
        const float alpha = mat_alpha(*S, m, u * m.tiling[0], v * m.tiling[1]);
        T = T * (1.0f - alpha);
        if (T > (eps_rule ? EPSILON : 0.0f)) return false;
        shadowed = true;
        return true;
    }
};

/* Shadow segments, lightSampling.glsl:108-144 with raySecondary.{rahit,rchit,rmiss}.glsl. */
template <int STACK, bool COUNT>
__device__ __forceinline__ f3 shadow_walk(const DScene &S, const JobView &J, f3 origin, f3 dir, float tmax_light,
                                          bool inside, uint32_t volIdx, uint2 *my, TraceCount &cnt, uint32_t &nseg) {
    const float tmin = 0.0001f;
    f3 T = {1, 1, 1};
    bool shadowed = false;
    float distanceT = tmax_light - tmin;
    const bool any_transparent = (J.scene_flags & SCENE_HAS_TRANSPARENT) != 0u;
    if (any_transparent && !(J.scene_flags & SCENE_HAS_VOLUME_CHANGE)) {
        /* No surface changes volume, so the reference's any-hit loop (raySecondary.rahit.glsl:31-72) is
         * order-independent: any opaque candidate shadows, transparent ones multiply by 1 - alpha, and
         * the walk stops once the product falls to EPSILON.  One walk, one segment. */
        ShadowAnyHit ah{&S, 1.0f, false, true};
        TraceHit h, hA;
        nseg++;
        trace_ray<MODE_ANYHIT, STACK, kTraceBlock, COUNT, ShadowAnyHit>(S, J.tlas_root, origin, dir, tmin, distanceT, h, hA, 0.f,
                                                                         0.f, 0u, 0u, my, cnt, &ah);
        if (ah.shadowed) return {0, 0, 0};
        f3 T1 = {ah.T, ah.T, ah.T};
        if (inside) {
            const float vtend = fminf((float)(uint32_t)J.zfar, distanceT);
            T1 = T1 * vol_transmittance(S, volIdx, tmin, vtend);
            if (!(max3(T1) > EPSILON)) return {0, 0, 0};
        }
        return T1;
    }
    for (uint32_t dd = 0; dd < J.depth; ++dd) {
        float vtmin = tmin;
        bool stop = false;
        TraceHit h, hA;
        if (!any_transparent) {
            nseg++;
            if (trace_ray<MODE_ANY, STACK, kTraceBlock, COUNT>(S, J.tlas_root, origin, dir, tmin, distanceT, h, hA, 0.f, 0.f, 0u,
                                                               0u, my, cnt)) {
                shadowed = true;
                stop = true;
            }
        } else {
            float pt = -1.0f;
            uint32_t pi = 0u, pp = 0u;
            bool accepted_change = false;
            for (;;) {
                nseg++;
                const bool found = trace_ray<MODE_ORDERED, STACK, kTraceBlock, COUNT>(S, J.tlas_root, origin, dir, tmin, distanceT, h,
                                                                                     hA, 0.f, pt, pi, pp, my, cnt);
                if (!found) break;
                const CandInfo c = cand_info(S, h, false);
                if (!c.transparent) {
                    shadowed = true;
                    stop = true;
                    break;
                }
                T = T * (1.0f - c.alpha);
                if (c.vol_change) {
                    accepted_change = true;
                    break;
                }
                if (max3(T) > EPSILON) {
                    pt = h.t;
                    pi = h.inst;
                    pp = h.prim;
                    continue;
                }
                shadowed = true;
                stop = true;
                break;
            }
            if (stop) break;
            if (accepted_change) {
                if (inside) {
                    T = T * vol_transmittance(S, volIdx, vtmin, h.t);
                    if (max3(T) < EPSILON) {
                        shadowed = true;
                        break;
                    }
                }
                vtmin = h.t;
                cross_volume_surface(S, h, dir, inside, volIdx, origin);
                distanceT -= vtmin;
                continue;
            }
        }
        if (!stop) {
            /* miss (raySecondary.rmiss.glsl) */
            stop = true;
            if (inside) {
                const float vtend = fminf((float)(uint32_t)J.zfar, distanceT);
                T = T * vol_transmittance(S, volIdx, vtmin, vtend);
                shadowed = !(max3(T) > EPSILON);
            }
        }
        distanceT -= vtmin;
        if (stop) break;
    }
    if (shadowed) T = {0, 0, 0};
    return T;
}

/* Emitter lookup along a BSDF direction, next_event_estimation.glsl:1-33 and rayNEE.{rahit,rchit,rmiss}.glsl. */
template <int STACK, bool COUNT>
__device__ __forceinline__ bool nee_walk(const DScene &S, const JobView &J, f3 origin, f3 dir, bool inside,
                                         uint32_t volIdx, uint2 *my, TraceCount &cnt, uint32_t &nseg, f3 &T, f3 &e,
                                         float &pdf) {
    const float tmin = 0.0001f;
    const float tmax = J.zfar;
    T = {1, 1, 1};
    for (uint32_t dd = 0; dd < J.depth; ++dd) {
        float pt = -1.0f;
        uint32_t pi = 0u, pp = 0u;
        TraceHit h, hA;
        bool crossed = false;
        for (;;) {
            nseg++;
            bool found;
            if (J.scene_flags & SCENE_HAS_TRANSPARENT)
                found = trace_ray<MODE_ORDERED, STACK, kTraceBlock, COUNT>(S, J.tlas_root, origin, dir, tmin, tmax, h, hA, 0.f, pt,
                                                                          pi, pp, my, cnt);
            else
                found = trace_ray<MODE_CLOSEST, STACK, kTraceBlock, COUNT>(S, J.tlas_root, origin, dir, tmin, tmax, h, hA, 0.f, 0.f,
                                                                          0u, 0u, my, cnt);
            if (!found) return false; /* rayNEE.rmiss.glsl */
            const CandInfo c = cand_info(S, h, true);
            if (isBlackEps(c.emissive, 0.05f)) {
                if (!c.transparent) return false;
                T = T * (1.0f - c.alpha);
                if (c.vol_change) {
                    crossed = true;
                    break;
                }
                pt = h.t;
                pi = h.inst;
                pp = h.prim;
                continue;
            }
            return nee_emitter(S, J, h, origin, dir, inside, volIdx, T, c.emissive, e, pdf);
        }
        if (crossed) {
            if (inside) {
                T = T * vol_transmittance(S, volIdx, tmin, h.t);
                if (max3(T) < EPSILON) return false;
            }
            cross_volume_surface(S, h, dir, inside, volIdx, origin);
        }
    }
    return false;
}

template <int STACK, bool COUNT, bool MULTI>
__global__ __launch_bounds__(kTraceBlock) void k_secondary(DScene S, RenderParams P, PathState st) {
    __shared__ uint2 stack[STACK * kTraceBlock];
    uint2 *my = stack + threadIdx.x;
    uint32_t nsh = 0, nne = 0;
    TraceCount cnt = {0, 0};
    uint32_t shard = wave_global_id() % kShards;
    bool done = false;
    for (;;) {
        /* one record per lane per round: these walks are rare and long */
        uint32_t r = 0;
        bool got = false;
        {
            /* every lane is idle here, so the refill threshold is met */
            uint32_t v = 0;
            got = sq_refill(P.sec, true, shard, done, v);
            r = v;
        }
        if (__ballot(got) == 0ull) {
            if (done) break;
            continue;
        }
        if (got) {
            const uint32_t kind = r % 3u;
            const uint32_t x = sec_ix(st, r);
            const float4 o4 = st.sec_o[x], d4 = st.sec_d[x], c4 = st.sec_c[x];
            const uint32_t vol = P.media ? (uint32_t)st.sec_v[x] : kInvalid;
            const bool inside = vol != kInvalid;
            const JobView &J = job_of<MULTI>(S, st, r / 3u);
            f3 res = {0, 0, 0};
            if (kind == 0u) {
                const f3 T = shadow_walk<STACK, COUNT>(S, J, ld3(o4), ld3(d4), o4.w, inside, vol, my, cnt, nsh);
                if (!isBlack(T)) res = ld3(c4) * T;
            } else {
                f3 T, e;
                float lpdf = 0.0f;
                if (nee_walk<STACK, COUNT>(S, J, ld3(o4), ld3(d4), inside, vol, my, cnt, nne, T, e, lpdf)) {
                    if (!isBlack(e)) res = PowerHeuristic(d4.w, lpdf) * T * e * ld3(c4);
                }
            }
            st.sec_c[x] = st4(res, 0.f);
        }
    }
    wave_add64(P.stats, S_SHADOW_SEC, nsh);
    wave_add64(P.stats, S_NEE, nne);
    if (COUNT) {
        wave_add64(P.stats, S_NODES_SEC, cnt.nodes);
        wave_add64(P.stats, S_TRIS_SEC, cnt.tris);
    }
}

/* ---------------------------------------------------------- k_shadow -- */
/* k_shadow's arguments in place: its queue is read where lanes refill.  Held in scalar registers it spilled 38 of them in
 * the batched kernel with alpha (8 this way): 24 jobs 66.3 -> 65.0 ms. */
struct TraceArgs {
    DScene S;
    RenderParams P;
    PathState st;
};
static_assert(sizeof(DScene) % alignof(RenderParams) == 0 && sizeof(RenderParams) % alignof(PathState) == 0,
              "laid out as the kernel's three arguments");
/* Shadow segments that end at the light or the first occluder
 * (lightSampling.glsl:108-144 when no surface changes volume): persistent
 * walk with lane refill; opaque scenes stop at the first hit, scenes with
 * transparent materials apply the any-hit product of 1 - alpha. */
template <int STACK, bool COUNT, bool ALPHA, bool MULTI>
__global__ __launch_bounds__(kTraceBlock) VVPT_TRACE_OCCUPANCY void k_shadow(DScene S, RenderParams P, PathState st) {
    __shared__ uint2 stack[(STACK + 3) * kTraceBlock]; /* the walk stack + the world ray */
    uint2 *my = stack + threadIdx.x;
    uint32_t nrays = 0;
    TraceCount cnt = {0, 0};
    Trav w;
    ShadowAnyHit ah{&S, 1.0f, false, true};
    bool active = false, done = false;
    uint32_t shard = wave_global_id() % kShards, r = 0;
    for (;;) {
        uint32_t v = 0;
        if (sq_refill(kernargs<TraceArgs>().P.shd, !active, shard, done, v) && !active) {
            r = v;
            const uint32_t x = sec_ix(st, r);
            const float4 o4 = st.sec_o[x], d4 = st.sec_d[x];
            /* record 0: light sample segment [1e-4, distance - 1e-4] (lightSampling.glsl:112-128);
             * record 1: passed surfaces in front of an emitter, [1e-4, o4.w] */
            const bool lightseg = (r % 3u) == 0u;
            trav_init<STACK, kTraceBlock>(w, my, job_of<MULTI>(S, st, r / 3u).tlas_root, ld3(o4), ld3(d4), 0.0001f, 0.0001f,
                      lightseg ? o4.w - 0.0001f : o4.w);
            ah.T = 1.0f;
            ah.shadowed = false;
            ah.eps_rule = lightseg;
            active = true;
            nrays++;
        }
        const unsigned long long am = __ballot(active);
        if (am == 0ull) {
            if (done) break;
            continue;
        }
        bool fin = false;
        if (active) {
            if (ALPHA)
                fin = trav_step<MODE_ANYHIT, STACK, kTraceBlock, COUNT, ShadowAnyHit>(w, S, my, cnt, &ah);
            else
                fin = trav_step<MODE_ANY, STACK, kTraceBlock, COUNT>(w, S, my, cnt);
        }
        if (fin) {
            const bool shadowed = ALPHA ? ah.shadowed : (w.hit.prim != kInvalid);
            f3 T = {0, 0, 0};
            if (!shadowed) {
                T = ALPHA ? mk(ah.T, ah.T, ah.T) : mk(1, 1, 1);
                const uint32_t vol = P.media ? (uint32_t)st.sec_v[sec_ix(st, r)] : kInvalid;
                if (vol != kInvalid) {
                    /* raySecondary.rmiss.glsl:24-42 */
                    const float vtend = fminf((float)(uint32_t)job_of<MULTI>(S, st, r / 3u).zfar, w.tmax);
                    T = T * vol_transmittance(S, vol, 0.0001f, vtend);
                    if (!(max3(T) > EPSILON)) T = {0, 0, 0};
                }
            }
            const uint32_t x = sec_ix(st, r);
            const float4 c4 = st.sec_c[x];
            st.sec_c[x] = st4(isBlack(T) ? mk(0, 0, 0) : ld3(c4) * T, 0.f);
            active = false;
        }
    }
    wave_add64(P.stats, S_SHADOW, nrays);
    if (COUNT) {
        wave_add64(P.stats, S_NODES_SHD, cnt.nodes);
        wave_add64(P.stats, S_TRIS_SHD, cnt.tris);
    }
}

/* Wall clock at the start of a batched render (the reference point of the jobs' completion times). */
__global__ void k_clock_stamp(unsigned long long *out) {
    if (threadIdx.x == 0u) *out = wall_clock64();
}

/* ------------------------------------------------- k_sample_sequence -- */
/* out[k * dims + d] = dimension d of sample first + k of one pixel's sequence (extended-mode sampler). */
__global__ void k_sample_sequence(uint32_t key, uint32_t first, uint32_t count, uint32_t dims, float *out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count * dims) return;
    out[i] = sampler_float(key, first + i / dims, i % dims);
}

/* ---------------------------------------------------------- k_resolve -- */
/* image = (first window ? 0 : image) + partial[b] for each batch b of the window, in batch order. */
__global__ void k_resolve(RenderParams P, JobView J, uint32_t nb, uint32_t first, float4 *outR, float4 *outA,
                          float4 *outN) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= J.npix) return;
    const size_t o = J.item_begin;
    f3 R = first ? mk(0.f, 0.f, 0.f) : ld3(outR[p]);
    for (uint32_t b = 0; b < nb; ++b) R = R + ld3(P.partR[o + (size_t)b * J.npix + p]);
    outR[p] = st4(R, 1.0f);
    if (P.aovs) {
        f3 A = first ? mk(0.f, 0.f, 0.f) : ld3(outA[p]), N = first ? mk(0.f, 0.f, 0.f) : ld3(outN[p]);
        for (uint32_t b = 0; b < nb; ++b) {
            A = A + ld3(P.partA[o + (size_t)b * J.npix + p]);
            N = N + ld3(P.partN[o + (size_t)b * J.npix + p]);
        }
        outA[p] = st4(A, 1.0f);
        outN[p] = st4(N, 1.0f);
    }
}

/* -------------------------------------------------- k_trace_primary -- */
template <int STACK>
__global__ __launch_bounds__(kTraceBlock) void k_trace_primary(DScene S, uint32_t W, uint32_t H, uint32_t seed,
                                                                 uint32_t *inst, uint32_t *prim, float *t, float *u,
                                                                 float *v) {
    __shared__ uint2 stack[STACK * kTraceBlock];
    uint2 *my = stack + threadIdx.x;
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= W * H) return;
    const uint32_t px = p % W, py = p / W;
    Rng rng = {initRNG(px, py, W, 0u, seed), 0u, 0u, false};
    f3 o, d;
    camera_ray(S.job, px, py, rng, o, d);
    TraceHit h, hA;
    TraceCount cnt = {0, 0};
    trace_ray<MODE_CLOSEST, STACK, kTraceBlock, false>(S, S.job.tlas_root, o, d, 0.001f, 10000.0f, h, hA, 0.f, 0.f, 0u, 0u,
                                                       my, cnt);
    inst[p] = h.inst;
    prim[p] = h.prim != kInvalid ? h.prim - S.insts[h.inst].idx_offset : kInvalid; /* the mesh's own index */
    t[p] = h.prim != kInvalid ? h.t : 0.0f;
    u[p] = h.prim != kInvalid ? h.u : 0.0f;
    v[p] = h.prim != kInvalid ? h.v : 0.0f;
}

}  // namespace vvpt
