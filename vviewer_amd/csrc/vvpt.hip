/*
 * vvpt.hip - C ABI of the gfx950 path tracer (include/vvpt.h).
 *
 * Host side of VulkanRendererPathTracing (src/lib/vengine/vulkan/renderers/
 * VulkanRendererPathTracing.cpp): scene upload and acceleration-structure
 * build (VulkanScene.cpp:306-381, VulkanAccelerationStructure.cpp), per-render
 * SceneData (:143-198), the batch loop (:791-901) as a wavefront loop over
 * work items, and readback (:903-956).
 */
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstddef>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/vvpt.h"
#include "bvh_build.h"
#include "denoise.h"
#include "lbvh_build.h"
#include "nrc_model.h"
#include "kernels.h"

using namespace vvpt;

static_assert(sizeof(vvpt_job) == 48 && offsetof(vvpt_job, d_radiance_rgba) == 32, "vvpt_job layout");
static_assert(sizeof(vvpt_tuning) == 12, "vvpt_tuning layout");
static_assert(sizeof(vvpt_options) == 48, "vvpt_options layout");

namespace {

struct DevBuf {
    void *p = nullptr;
    size_t bytes = 0;
};

struct SceneHost {
    bool valid = false;
    uint32_t num_instances = 0, num_triangles = 0;
    uint32_t tlas_nodes = 0, blas_nodes = 0, max_depth = 0;
    uint32_t scene_flags = 0;
    bool textured = false; /* some material binds a texture of its own to a slot other than alpha */
    bool walks = false; /* some material is transparent (of whatever type) or some instance changes volume */
    uint32_t num_lights = 0;
    uint32_t cube_w = 0;
    uint32_t env_mw = 0, env_mh = 0;
    float scene_lo[3] = {0, 0, 0}, scene_hi[3] = {1, 1, 1}; /* union of the instance boxes */
    uint32_t tlas_root = 0;
    vvpt_camera cam{};
    vvpt_environment env{};
    std::vector<vvpt_material> mats_desc;
    /* scene parts (vvpt_set_scenes): each keeps its own TLAS, light list and camera */
    struct Part {
        uint32_t tlas_root, light_begin, num_lights;
        uint32_t scene_flags; /* SCENE_HAS_* of the part alone */
        uint32_t mat_begin;   /* the part's first material in the merged description (its camera's volume is offset) */
        vvpt_camera cam;
    };
    std::vector<Part> parts;
};

/* Where each part of a merged scene description starts. */
struct PartRange {
    uint32_t inst_begin, inst_count;   /* instances of the part in the merged description */
    uint32_t light_begin, light_count; /* its point / directional lights */
    vvpt_camera cam;
    uint32_t mat_begin, mat_count;     /* its materials */
};

}  // namespace

struct vvpt_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    std::string last_error;
    std::atomic<bool> busy{false};
    std::atomic<float> progress{0.0f};
    SceneHost sh;
    /* scene buffers */
    DevBuf nodes, tris, tlas_leaf, insts, triverts, instmats, mats, texs, tex8, texf, lights, cube, srgb;
    DevBuf env_prob, env_alias, env_cpdf; /* environment importance grid (extended mode) */
    DevBuf nrcbuf;                        /* radiance-cache render buffers */
    DevBuf jobbuf;                        /* batched render: job table, completion ticks, remaining items */
    DevBuf dnbuf, dnio;                   /* denoiser: ping-pong images; host-call staging */
    /* render buffers (grown on demand) */
    DevBuf state, queues, counters, stats, partials, outputs;
    uint32_t *h_counters = nullptr; /* pinned copy of the counter block */
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    std::vector<hipEvent_t> kev; /* per-launch timing events (VVPT_FLAG_KERNEL_TIMING) */
    uint32_t builder = VVPT_BUILDER_SAH;
    NrcModel *nrc = nullptr; /* neural radiance cache, created on first use */
    vvpt_tuning tune{1u << 25, 12u, 64u}; /* launch shape (vvpt_set_tuning / vvpt_autotune) */
    vvpt_options opt{};                   /* render options (vvpt_set_options); zero fields are defaults */
    uint32_t cus = 0;                    /* compute units of the device */
};

namespace {

vvpt_status set_err(vvpt_ctx *c, vvpt_status s, const std::string &msg) {
    if (c) c->last_error = msg;
    return s;
}

/* One call at a time may change or use a context's device state: every entry point that does takes the context
 * for its whole duration (a second caller gets VVPT_BUSY, like the reference's render guard,
 * VulkanRendererPathTracing.cpp:123-124); progress, errors and getters stay readable. */
struct BusyGuard {
    vvpt_ctx *c;
    bool ok;
    explicit BusyGuard(vvpt_ctx *cc) : c(cc) {
        bool expected = false;
        ok = c->busy.compare_exchange_strong(expected, true);
    }
    ~BusyGuard() {
        if (ok) c->busy.store(false);
    }
};

#define VVPT_TAKE(ctx)                                                                                      \
    BusyGuard _take(ctx);                                                                                   \
    if (!_take.ok) return set_err(ctx, VVPT_BUSY, "render in progress")

#define HIP_TRY(ctx, expr)                                                                                  \
    do {                                                                                                    \
        hipError_t _e = (expr);                                                                             \
        if (_e != hipSuccess)                                                                               \
            return set_err(ctx, _e == hipErrorOutOfMemory ? VVPT_OOM : VVPT_DEVICE_LOST,                    \
                           std::string(#expr) + ": " + hipGetErrorString(_e));                              \
    } while (0)

hipError_t upload(DevBuf &b, const void *src, size_t bytes, hipStream_t s) {
    if (b.p) {
        (void)hipFree(b.p);
        b.p = nullptr;
        b.bytes = 0;
    }
    size_t n = std::max<size_t>(bytes, 16);
    hipError_t e = hipMalloc(&b.p, n);
    if (e != hipSuccess) return e;
    b.bytes = n;
    if (bytes) {
        e = hipMemcpyAsync(b.p, src, bytes, hipMemcpyHostToDevice, s);
        if (e != hipSuccess) return e;
        e = hipStreamSynchronize(s);
    }
    return e;
}
hipError_t ensure(DevBuf &b, size_t bytes) {
    if (b.bytes >= bytes && b.p) return hipSuccess;
    if (b.p) (void)hipFree(b.p);
    b.p = nullptr;
    b.bytes = 0;
    hipError_t e = hipMalloc(&b.p, bytes);
    if (e == hipSuccess) b.bytes = bytes;
    return e;
}
void release(DevBuf &b) {
    if (b.p) (void)hipFree(b.p);
    b.p = nullptr;
    b.bytes = 0;
}

/* Inverse of a column-major 4x4 in float, rounded as glm::inverse rounds it (the reference inverts its
 * camera matrices with glm on the host, core/Camera.cpp:43-47, VulkanRendererPathTracing.cpp:155):
 * cofactor (row c, column j) expanded along the first remaining column, each 2x2 minor taken as
 * m(p,r)*m(q,s) - m(q,r)*m(p,s), the three terms summed left to right; determinant from the first
 * column as (t0 + t1) + (t2 + t3); every cofactor times 1/det. */
bool inverse4_glm(const float *a, float *out) {
#pragma clang fp contract(off)
    auto m = [a](int c, int r) { return a[c * 4 + r]; };
    auto minor2 = [&](int p, int q, int r, int s) { return m(p, r) * m(q, s) - m(q, r) * m(p, s); };
    float cof[4][4];
    for (int c = 0; c < 4; ++c) {
        int rows[3], n = 0;
        for (int r = 0; r < 4; ++r)
            if (r != c) rows[n++] = r;
        for (int j = 0; j < 4; ++j) {
            int cols[3], k = 0;
            for (int q = 0; q < 4; ++q)
                if (q != j) cols[k++] = q;
            const float t = m(cols[0], rows[0]) * minor2(cols[1], cols[2], rows[1], rows[2]) -
                            m(cols[0], rows[1]) * minor2(cols[1], cols[2], rows[0], rows[2]) +
                            m(cols[0], rows[2]) * minor2(cols[1], cols[2], rows[0], rows[1]);
            cof[c][j] = ((c + j) & 1) ? -t : t;
        }
    }
    const float det = (m(0, 0) * cof[0][0] + m(0, 1) * cof[1][0]) + (m(0, 2) * cof[2][0] + m(0, 3) * cof[3][0]);
    if (!(det != 0.0f) || !std::isfinite(det)) return false;
    const float rdet = 1.0f / det;
    for (int c = 0; c < 4; ++c)
        for (int j = 0; j < 4; ++j) out[c * 4 + j] = cof[c][j] * rdet;
    return true;
}

/* double-precision inverse of a 4x4 column-major matrix */
bool inverse4(const double *a, double *out) {
    double m[4][8];
    for (int r = 0; r < 4; ++r)
        for (int c = 0; c < 4; ++c) {
            m[r][c] = a[c * 4 + r];
            m[r][c + 4] = r == c ? 1.0 : 0.0;
        }
    for (int col = 0; col < 4; ++col) {
        int piv = col;
        for (int r = col + 1; r < 4; ++r)
            if (std::fabs(m[r][col]) > std::fabs(m[piv][col])) piv = r;
        if (m[piv][col] == 0.0) return false;
        if (piv != col)
            for (int c = 0; c < 8; ++c) std::swap(m[piv][c], m[col][c]);
        double inv = 1.0 / m[col][col];
        for (int c = 0; c < 8; ++c) m[col][c] *= inv;
        for (int r = 0; r < 4; ++r)
            if (r != col) {
                double f = m[r][col];
                if (f != 0.0)
                    for (int c = 0; c < 8; ++c) m[r][c] -= f * m[col][c];
            }
    }
    for (int r = 0; r < 4; ++r)
        for (int c = 0; c < 4; ++c) out[c * 4 + r] = m[r][c + 4];
    return true;
}

float srgb_to_linear(float c) { return c <= 0.04045f ? c / 12.92f : std::pow((c + 0.055f) / 1.055f, 2.4f); }

/* equirect uv of a direction, environmentMap.glsl:1-10 */
void equirect_uv(const float *v, float &u, float &w) {
    float x = std::atan2(v[2], v[0]) * 0.1591f + 0.5f;
    w = std::asin(v[1]) * 0.3183f + 0.5f;
    x = x + 0.25f;
    u = x - std::floor(x);
}

struct HostTex {
    uint32_t w, h, fmt;
    const uint8_t *b8;
    const float *f;
};
void host_tex_sample(const HostTex &t, float u, float v, float *out) {
    auto fetch = [&](uint32_t x, uint32_t y, float *c) {
        size_t k = (size_t)y * t.w + x;
        if (t.fmt == VVPT_TEXTURE_RGBA32F) {
            for (int j = 0; j < 4; ++j) c[j] = t.f[4 * k + j];
        } else {
            for (int j = 0; j < 4; ++j) {
                float f = t.b8[4 * k + j] / 255.0f;
                c[j] = (t.fmt == VVPT_TEXTURE_RGBA8_SRGB && j < 3) ? srgb_to_linear(f) : f;
            }
        }
    };
    if (t.w == 1 && t.h == 1) {
        fetch(0, 0, out);
        return;
    }
    float x = u * t.w - 0.5f, y = v * t.h - 0.5f;
    float fx = std::floor(x), fy = std::floor(y);
    float a = x - fx, b = y - fy;
    auto wrap = [](long long i, uint32_t n) {
        long long m = i % (long long)n;
        return (uint32_t)(m < 0 ? m + n : m);
    };
    uint32_t x0 = wrap((long long)fx, t.w), x1 = wrap((long long)fx + 1, t.w), y0 = wrap((long long)fy, t.h),
             y1 = wrap((long long)fy + 1, t.h);
    float c00[4], c10[4], c01[4], c11[4];
    fetch(x0, y0, c00);
    fetch(x1, y0, c10);
    fetch(x0, y1, c01);
    fetch(x1, y1, c11);
    float w00 = (1 - a) * (1 - b), w10 = a * (1 - b), w01 = (1 - a) * b, w11 = a * b;
    for (int j = 0; j < 4; ++j) out[j] = c00[j] * w00 + c10[j] * w10 + c01[j] * w01 + c11[j] * w11;
}

/* cube face direction of (s,t) in [0,1]^2 (Vulkan cube-map face orientation) */
void cube_dir(int f, float s, float t, float *d) {
    float sc = 2.0f * s - 1.0f, tc = 2.0f * t - 1.0f;
    float x, y, z;
    switch (f) {
        case 0: x = 1.0f; y = -tc; z = -sc; break;
        case 1: x = -1.0f; y = -tc; z = sc; break;
        case 2: x = sc; y = 1.0f; z = tc; break;
        case 3: x = sc; y = -1.0f; z = -tc; break;
        case 4: x = sc; y = -tc; z = 1.0f; break;
        default: x = -sc; y = -tc; z = -1.0f; break;
    }
    float l = std::sqrt(x * x + y * y + z * z);
    d[0] = x / l;
    d[1] = y / l;
    d[2] = z / l;
}

bool material_is_emissive(const vvpt_material &m) {
    /* Material::isEmissive, core/Material.cpp:85-88,140-143 */
    return m.emissive[3] > 1.1920929e-07f &&
           !(std::fabs(m.emissive[0]) <= 0.01f && std::fabs(m.emissive[1]) <= 0.01f && std::fabs(m.emissive[2]) <= 0.01f);
}

/* Counter block: count and fetch counters of the queues, and the work-item counters. */
enum : uint32_t { CB_EXT0 = 0, CB_EXT1 = 2, CB_SEC = 4, CB_SHD = 6, CB_ITEMS = 8, CB_NRCQ = 9, CB_N = 11 };
constexpr size_t kCounterBytes = (size_t)CB_N * kShards * kPad * sizeof(uint32_t);

/* The environment importance grid of the extended mode: cell weights from the cube map on the device
 * (k_env_importance), a floor of 1 % of the mean radiance so that every direction keeps some density, and the
 * alias table on the host. */
std::string build_env_importance(vvpt_ctx *c, uint32_t cube_w) {
    constexpr uint32_t kMW = 1024, kMH = 512;
    const uint32_t n = kMW * kMH;
    DScene S;
    std::memset(&S, 0, sizeof(S));
    S.cube = (const float4 *)c->cube.p;
    S.cube_w = cube_w;
    DevBuf wbuf;
    if (ensure(wbuf, n * sizeof(float)) != hipSuccess) return "allocation";
    hipLaunchKernelGGL(k_env_importance, dim3((n + 255) / 256), dim3(256), 0, c->stream, S, kMW, kMH, (float *)wbuf.p);
    std::vector<float> wf(n);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(wf.data(), wbuf.p, n * sizeof(float), hipMemcpyDeviceToHost, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    release(wbuf);
    if (e != hipSuccess) return hipGetErrorString(e);
    double mean_rad = 0.0;
    std::vector<double> sinw(n);
    for (uint32_t i = 0; i < n; ++i) {
        sinw[i] = std::sin(((double)(i / kMW) + 0.5) * M_PI / kMH);
        mean_rad += sinw[i] > 0 ? wf[i] / sinw[i] : 0.0;
    }
    mean_rad /= n;
    if (!(mean_rad > 0.0)) return "";
    std::vector<double> w(n);
    for (uint32_t i = 0; i < n; ++i) w[i] = (double)wf[i] + 0.01 * mean_rad * sinw[i];
    std::vector<float> prob, cpdf;
    std::vector<uint32_t> alias;
    build_alias(w, prob, alias, cpdf);
    if ((e = upload(c->env_prob, prob.data(), n * sizeof(float), c->stream)) != hipSuccess) return hipGetErrorString(e);
    if ((e = upload(c->env_alias, alias.data(), n * sizeof(uint32_t), c->stream)) != hipSuccess) return hipGetErrorString(e);
    if ((e = upload(c->env_cpdf, cpdf.data(), n * sizeof(float), c->stream)) != hipSuccess) return hipGetErrorString(e);
    c->sh.env_mw = kMW;
    c->sh.env_mh = kMH;
    return "";
}

/* Build one wide BVH over `boxes` with the context's builder and append it to nodes / refs (child_base and
 * leaf_base made absolute).  Returns an empty string or the failing step. */
std::string build_bvh(vvpt_ctx *c, const std::vector<Box3> &boxes, int max_leaf, std::vector<WideNode> &nodes,
                      std::vector<uint32_t> &refs, WideBuildResult &r) {
    if (c->builder != VVPT_BUILDER_LBVH) {
        r = build_wide_bvh(boxes, max_leaf, nodes, refs);
        return "";
    }
    std::vector<float> b6(6 * boxes.size());
    for (size_t i = 0; i < boxes.size(); ++i)
        for (int a = 0; a < 3; ++a) {
            b6[6 * i + a] = boxes[i].lo[a];
            b6[6 * i + 3 + a] = boxes[i].hi[a];
        }
    LbvhOutput o;
    const std::string err = lbvh_build_device(b6.data(), (uint32_t)boxes.size(), (uint32_t)max_leaf, false, c->stream, o);
    if (!err.empty()) return err;
    const uint32_t nbase = (uint32_t)nodes.size(), rbase = (uint32_t)refs.size();
    for (WideNode w : o.nodes) {
        w.child_base += nbase;
        w.leaf_base += rbase;
        nodes.push_back(w);
    }
    refs.insert(refs.end(), o.leaf_refs.begin(), o.leaf_refs.end());
    r.root = nbase;
    r.depth = o.depth;
    return "";
}

}  // namespace

extern "C" {

uint32_t vvpt_abi_version(void) { return VVPT_ABI_VERSION; }

vvpt_status vvpt_create(vvpt_ctx **out, int hip_device) {
    if (!out) return VVPT_INVALID;
    *out = nullptr;
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) return VVPT_UNSUPPORTED;
    if (hip_device < 0 || hip_device >= n) return VVPT_INVALID;
    vvpt_ctx *c = new vvpt_ctx();
    c->device = hip_device;
    if (hipSetDevice(hip_device) != hipSuccess) {
        delete c;
        return VVPT_DEVICE_LOST;
    }
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, hip_device) != hipSuccess) {
        delete c;
        return VVPT_DEVICE_LOST;
    }
    if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) {
        delete c;
        return VVPT_UNSUPPORTED;
    }
    c->cus = (uint32_t)prop.multiProcessorCount;
    if (hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess ||
        hipHostMalloc((void **)&c->h_counters, kCounterBytes, hipHostMallocDefault) != hipSuccess ||
        hipEventCreate(&c->ev0) != hipSuccess || hipEventCreate(&c->ev1) != hipSuccess) {
        vvpt_destroy(c);
        return VVPT_DEVICE_LOST;
    }
    float lut[256];
    for (int i = 0; i < 256; ++i) lut[i] = srgb_to_linear(i / 255.0f);
    if (upload(c->srgb, lut, sizeof(lut), c->stream) != hipSuccess) {
        vvpt_destroy(c);
        return VVPT_DEVICE_LOST;
    }
    /* device address of the allocation-free denoise's fixed scratch on this device (the device is current) */
    if (!denoise_scratch_init(hip_device).empty()) {
        vvpt_destroy(c);
        return VVPT_DEVICE_LOST;
    }
    *out = c;
    return VVPT_OK;
}

void vvpt_destroy(vvpt_ctx *c) {
    if (!c) return;
    (void)hipSetDevice(c->device);
    (void)hipStreamSynchronize(c->stream);
    DevBuf *bufs[] = {&c->nodes, &c->tris, &c->tlas_leaf, &c->insts, &c->triverts, &c->instmats, &c->mats,
                      &c->texs, &c->tex8, &c->texf, &c->lights, &c->cube, &c->srgb, &c->env_prob, &c->env_alias, &c->env_cpdf, &c->nrcbuf, &c->jobbuf, &c->dnbuf, &c->dnio, &c->state,
                      &c->queues, &c->counters, &c->stats, &c->partials, &c->outputs};
    for (DevBuf *b : bufs) release(*b);
    if (c->h_counters) (void)hipHostFree(c->h_counters);
    for (hipEvent_t e : c->kev) (void)hipEventDestroy(e);
    if (c->ev0) (void)hipEventDestroy(c->ev0);
    if (c->ev1) (void)hipEventDestroy(c->ev1);
    delete c->nrc;
    if (c->stream) (void)hipStreamDestroy(c->stream);
    delete c;
}

int vvpt_is_enabled(const vvpt_ctx *c) { return c != nullptr; }

float vvpt_progress(const vvpt_ctx *c) { return c ? c->progress.load() : 0.0f; }

const char *vvpt_last_error(const vvpt_ctx *c) { return c ? c->last_error.c_str() : "null context"; }

static vvpt_status set_scene_parts(vvpt_ctx *c, const vvpt_scene_desc *D, const std::vector<PartRange> &parts) {
    c->sh = SceneHost();
    /* validate */
    for (uint32_t i = 0; i < D->num_instances; ++i) {
        const vvpt_instance &in = D->instances[i];
        if (in.mesh >= D->num_meshes || in.material >= D->num_materials)
            return set_err(c, VVPT_INVALID, "instance references a missing mesh or material");
        if ((in.front_volume >= 0 && (uint32_t)in.front_volume >= D->num_materials) ||
            (in.back_volume >= 0 && (uint32_t)in.back_volume >= D->num_materials))
            return set_err(c, VVPT_INVALID, "instance references a missing volume material");
    }
    for (uint32_t i = 0; i < D->num_meshes; ++i) {
        const vvpt_mesh &m = D->meshes[i];
        for (size_t k = 0; k < (size_t)m.num_triangles * 3; ++k)
            if (m.indices[k] >= m.num_vertices) return set_err(c, VVPT_INVALID, "mesh index out of range");
    }
    for (uint32_t i = 0; i < D->num_textures; ++i) {
        const vvpt_texture &t = D->textures[i];
        if (t.width == 0 || t.height == 0 || !t.data || t.format > VVPT_TEXTURE_RGBA32F)
            return set_err(c, VVPT_INVALID, "bad texture");
    }

    /* textures: 0 white, 1 whiteColor, 2 normalmapdefault (core/Image.hpp:40-90) */
    std::vector<DTexture> texs;
    std::vector<uint32_t> tex8 = {0xFFFFFFFFu, 0xFFFFFFFFu, 0xFFFF8080u};
    std::vector<float4> texf;
    texs.push_back({0, 1, 1, 0});
    texs.push_back({1, 1, 1, 1});
    texs.push_back({2, 1, 1, 0});
    for (uint32_t i = 0; i < D->num_textures; ++i) {
        const vvpt_texture &t = D->textures[i];
        size_t n = (size_t)t.width * t.height;
        if (t.format == VVPT_TEXTURE_RGBA32F) {
            texs.push_back({(uint32_t)texf.size(), t.width, t.height, t.format});
            const float *f = (const float *)t.data;
            for (size_t k = 0; k < n; ++k) texf.push_back(make_float4(f[4 * k], f[4 * k + 1], f[4 * k + 2], f[4 * k + 3]));
        } else {
            texs.push_back({(uint32_t)tex8.size(), t.width, t.height, t.format});
            const uint32_t *b = (const uint32_t *)t.data;
            tex8.insert(tex8.end(), b, b + n);
        }
    }
    /* materials */
    std::vector<DMaterial> mats(D->num_materials);
    bool any_transparent = false;
    std::vector<uint8_t> mat_transparent(D->num_materials, 0);
    const uint32_t defaults[7] = {1, 0, 0, 0, 1, 2, 0}; /* VulkanMaterial.cpp:46-52 */
    for (uint32_t i = 0; i < D->num_materials; ++i) {
        const vvpt_material &m = D->materials[i];
        DMaterial &x = mats[i];
        std::memset(&x, 0, sizeof(x));
        std::memcpy(x.albedo, m.albedo, 16);
        x.mra[0] = m.metallic;
        x.mra[1] = m.roughness;
        x.mra[2] = m.ao;
        x.mra[3] = m.transparent;
        std::memcpy(x.emissive, m.emissive, 16);
        const int32_t ids[7] = {m.tex_albedo, m.tex_metallic, m.tex_roughness, m.tex_ao, m.tex_emissive, m.tex_normal, m.tex_alpha};
        uint32_t t[7];
        for (int k = 0; k < 7; ++k) t[k] = (ids[k] >= 0 && (uint32_t)ids[k] < D->num_textures) ? (uint32_t)ids[k] + 3 : defaults[k];
        x.tex1[0] = t[0];
        x.tex1[1] = t[1];
        x.tex1[2] = t[2];
        x.tex1[3] = t[3];
        x.tex2[0] = t[4];
        x.tex2[1] = t[5];
        x.tex2[2] = 0;
        x.tex2[3] = t[6];
        x.tiling[0] = m.uv_tiling[0];
        x.tiling[1] = m.uv_tiling[1];
        x.tiling[2] = (float)m.type;
        bool em = m.emissive[3] != 0.0f && (m.emissive[0] != 0.0f || m.emissive[1] != 0.0f || m.emissive[2] != 0.0f);
        x.flags = (em ? 1u : 0u) | (m.transparent > 0.0f ? 2u : 0u) | (m.type == VVPT_MATERIAL_VOLUME ? 4u : 0u);
        if (m.type != VVPT_MATERIAL_VOLUME && m.transparent > 0.0f) any_transparent = true, mat_transparent[i] = 1;
    }
    /* meshes: vertices, indices, BLAS */
    std::vector<DVertex> verts, tri_verts;
    std::vector<uint32_t> indices;
    std::vector<WideNode> nodes;
    std::vector<LeafTri> leaf_tris;
    std::vector<uint32_t> blas_root(D->num_meshes), vtx_off(D->num_meshes), idx_off(D->num_meshes);
    std::vector<Box3> mesh_box(D->num_meshes);
    uint32_t max_blas_depth = 0;
    for (uint32_t i = 0; i < D->num_meshes; ++i) {
        const vvpt_mesh &m = D->meshes[i];
        vtx_off[i] = (uint32_t)verts.size();
        idx_off[i] = (uint32_t)(indices.size() / 3);
        for (uint32_t k = 0; k < m.num_vertices; ++k) {
            const vvpt_vertex &s = m.vertices[k];
            DVertex v;
            v.px = s.position[0]; v.py = s.position[1]; v.pz = s.position[2]; v.u = s.uv[0];
            v.v = s.uv[1]; v.nx = s.normal[0]; v.ny = s.normal[1]; v.nz = s.normal[2];
            v.tx = s.tangent[0]; v.ty = s.tangent[1]; v.tz = s.tangent[2]; v.pad0 = 0.f;
            v.bx = s.bitangent[0]; v.by = s.bitangent[1]; v.bz = s.bitangent[2]; v.pad1 = 0.f;
            verts.push_back(v);
        }
        indices.insert(indices.end(), m.indices, m.indices + 3 * (size_t)m.num_triangles);
        for (size_t q = 0; q < 3 * (size_t)m.num_triangles; ++q) tri_verts.push_back(verts[vtx_off[i] + m.indices[q]]);
        std::vector<Box3> boxes(m.num_triangles);
        for (uint32_t p = 0; p < m.num_triangles; ++p)
            for (int k = 0; k < 3; ++k) boxes[p].grow(m.vertices[m.indices[3 * p + k]].position);
        for (const Box3 &b : boxes) mesh_box[i].grow(b);
        std::vector<uint32_t> refs;
        WideBuildResult r;
        const std::string berr = build_bvh(c, boxes, 3, nodes, refs, r);
        if (!berr.empty()) return set_err(c, VVPT_DEVICE_LOST, "BLAS build: " + berr);
        /* leaf references become absolute leaf-triangle records */
        uint32_t base = (uint32_t)leaf_tris.size();
        for (uint32_t p : refs) {
            LeafTri t;
            const float *a = m.vertices[m.indices[3 * p]].position, *b = m.vertices[m.indices[3 * p + 1]].position,
                        *cc = m.vertices[m.indices[3 * p + 2]].position;
            for (int k = 0; k < 3; ++k) {
                t.v0[k] = a[k];
                t.e1[k] = b[k] - a[k];
                t.e2[k] = cc[k] - a[k];
            }
            t.prim = idx_off[i] + p; /* global triangle index: the shading data of the hit is addressed by it */
            t.pad0 = t.pad1 = 0;
            leaf_tris.push_back(t);
        }
        /* shift this BLAS's leaf bases into the global leaf-triangle array */
        for (uint32_t nidx = r.root; nidx < nodes.size(); ++nidx) nodes[nidx].leaf_base += base;
        blas_root[i] = r.root;
        max_blas_depth = std::max(max_blas_depth, r.depth);
        c->sh.num_triangles += m.num_triangles;
    }
    c->sh.blas_nodes = (uint32_t)nodes.size();
    /* instances and TLAS */
    std::vector<DInstance> insts(D->num_instances);
    std::vector<Box3> iboxes(D->num_instances);
    bool any_volume_change = false;
    for (uint32_t i = 0; i < D->num_instances; ++i) {
        const vvpt_instance &s = D->instances[i];
        DInstance &x = insts[i];
        std::memset(&x, 0, sizeof(x));
        std::memcpy(x.o2w, s.transform, 48);
        double a[16] = {0}, inv[16];
        for (int r = 0; r < 3; ++r)
            for (int cc = 0; cc < 4; ++cc) a[cc * 4 + r] = s.transform[r * 4 + cc];
        a[15] = 1.0;
        if (!inverse4(a, inv)) return set_err(c, VVPT_INVALID, "singular instance transform");
        for (int r = 0; r < 3; ++r)
            for (int cc = 0; cc < 4; ++cc) x.w2o[r * 4 + cc] = (float)inv[cc * 4 + r];
        x.blas_root = blas_root[s.mesh];
        x.material = s.material;
        x.idg = (float)s.front_volume;
        x.idb = (float)s.back_volume;
        if (s.front_volume != s.back_volume) any_volume_change = true;
        x.vtx_offset = vtx_off[s.mesh];
        x.idx_offset = idx_off[s.mesh];
        x.ntri = D->meshes[s.mesh].num_triangles;
        {
            const vvpt_material &mm = D->materials[s.material];
            const bool em = mm.emissive[3] != 0.0f && (mm.emissive[0] != 0.0f || mm.emissive[1] != 0.0f || mm.emissive[2] != 0.0f);
            x.flags = (mm.transparent >= 0.99f ? INST_TRANSPARENT : 0u) | (mm.transparent > 0.0f ? INST_ALPHA_TEST : 0u) |
                      (s.front_volume != s.back_volume ? INST_VOL_CHANGE : 0u) | (em ? INST_EMISSIVE : 0u);
            if ((x.flags & INST_TRANSPARENT) && !em && s.front_volume == s.back_volume) x.flags |= INST_NEE_PASS;
        }
        const vvpt_mesh &m = D->meshes[s.mesh];
        for (uint32_t k = 0; k < m.num_vertices; ++k) {
            const float *p = m.vertices[k].position;
            float w[3];
            for (int r = 0; r < 3; ++r)
                w[r] = s.transform[r * 4] * p[0] + s.transform[r * 4 + 1] * p[1] + s.transform[r * 4 + 2] * p[2] +
                       s.transform[r * 4 + 3];
            iboxes[i].grow(w);
        }
        /* pad by a relative epsilon: the world box is made of rounded transforms */
        for (int r = 0; r < 3; ++r) {
            float e = 1e-5f * std::max(1.0f, std::max(std::fabs(iboxes[i].lo[r]), std::fabs(iboxes[i].hi[r])));
            iboxes[i].lo[r] -= e;
            iboxes[i].hi[r] += e;
        }
    }
    /* one TLAS per part over its instances; leaf references are global instance indices */
    std::vector<uint32_t> tlas_refs;
    size_t tlas_first = nodes.size();
    std::vector<uint32_t> part_root(parts.size());
    for (size_t pi = 0; pi < parts.size(); ++pi) {
        const PartRange &pr = parts[pi];
        std::vector<Box3> pboxes(iboxes.begin() + pr.inst_begin, iboxes.begin() + pr.inst_begin + pr.inst_count);
        std::vector<uint32_t> refs;
        WideBuildResult tr;
        const std::string terr = build_bvh(c, pboxes, 1, nodes, refs, tr);
        if (!terr.empty()) return set_err(c, VVPT_DEVICE_LOST, "TLAS build: " + terr);
        const uint32_t rbase = (uint32_t)tlas_refs.size();
        for (size_t k = (size_t)tr.root; k < nodes.size(); ++k) nodes[k].leaf_base += rbase;
        for (uint32_t r : refs) tlas_refs.push_back(r + pr.inst_begin);
        part_root[pi] = tr.root;
        c->sh.max_depth = std::max(c->sh.max_depth, tr.depth + max_blas_depth);
    }
    c->sh.tlas_nodes = (uint32_t)(nodes.size() - tlas_first);
    c->sh.tlas_root = part_root[0];
    {
        Box3 all;
        for (const Box3 &b : iboxes) all.grow(b);
        if (all.valid())
            for (int a = 0; a < 3; ++a) {
                c->sh.scene_lo[a] = all.lo[a];
                c->sh.scene_hi[a] = all.hi[a];
            }
    }
    /* lights of each part: point/directional, then mesh lights in instance order (VulkanInstances.cpp:71-108) */
    std::vector<DLight> lights;
    for (size_t pi = 0; pi < parts.size(); ++pi) {
        const PartRange &pr = parts[pi];
        SceneHost::Part part;
        part.tlas_root = part_root[pi];
        part.light_begin = (uint32_t)lights.size();
        part.cam = pr.cam;
        part.mat_begin = pr.mat_begin;
        part.scene_flags = 0u;
        for (uint32_t i = pr.mat_begin; i < pr.mat_begin + pr.mat_count; ++i)
            if (mat_transparent[i]) part.scene_flags |= SCENE_HAS_TRANSPARENT;
        for (uint32_t i = pr.inst_begin; i < pr.inst_begin + pr.inst_count; ++i)
            if (D->instances[i].front_volume != D->instances[i].back_volume) part.scene_flags |= SCENE_HAS_VOLUME_CHANGE;
        for (uint32_t i = pr.light_begin; i < pr.light_begin + pr.light_count; ++i) {
            const vvpt_light &l = D->lights[i];
            DLight x;
            std::memset(&x, 0, sizeof(x));
            x.type = l.type;
            x.intensity = l.color[3];
            std::memcpy(x.color, l.color, 16);
            x.position[0] = l.position[0];
            x.position[1] = l.position[1];
            x.position[2] = l.position[2];
            lights.push_back(x);
        }
        for (uint32_t i = pr.inst_begin; i < pr.inst_begin + pr.inst_count; ++i) {
            const vvpt_material &m = D->materials[D->instances[i].material];
            if (m.type == VVPT_MATERIAL_VOLUME || !material_is_emissive(m)) continue;
            DLight x;
            std::memset(&x, 0, sizeof(x));
            x.type = 2;
            x.inst = i;
            lights.push_back(x);
        }
        part.num_lights = (uint32_t)lights.size() - part.light_begin;
        c->sh.parts.push_back(part);
    }
    /* environment cube map (VulkanRendererSkybox.cpp:98-140, skyboxCubemapWrite.frag.glsl:12-15) */
    std::vector<float4> cube;
    uint32_t cube_w = 0;
    int et = D->environment.equirect_texture;
    if (et >= 0 && (uint32_t)et < D->num_textures) {
        const vvpt_texture &t = D->textures[et];
        HostTex E{t.width, t.height, t.format, (const uint8_t *)t.data, (const float *)t.data};
        cube_w = std::max(1u, std::min(t.width / 4, 1080u));
        cube.resize((size_t)6 * cube_w * cube_w);
        for (int f = 0; f < 6; ++f)
            for (uint32_t y = 0; y < cube_w; ++y)
                for (uint32_t x = 0; x < cube_w; ++x) {
                    float d[3], u, w, o[4];
                    cube_dir(f, (x + 0.5f) / cube_w, (y + 0.5f) / cube_w, d);
                    equirect_uv(d, u, w);
                    host_tex_sample(E, u, w, o);
                    cube[(size_t)f * cube_w * cube_w + (size_t)y * cube_w + x] = make_float4(o[0], o[1], o[2], o[3]);
                }
    }
    hipStream_t s = c->stream;
    HIP_TRY(c, upload(c->nodes, nodes.data(), nodes.size() * sizeof(WideNode), s));
    HIP_TRY(c, upload(c->tris, leaf_tris.data(), leaf_tris.size() * sizeof(LeafTri), s));
    std::vector<TlasLeaf> tlas_leaf(tlas_refs.size());
    for (size_t k = 0; k < tlas_refs.size(); ++k) {
        const DInstance &x = insts[tlas_refs[k]];
        TlasLeaf &l = tlas_leaf[k];
        std::memcpy(l.w2o, x.w2o, sizeof(l.w2o));
        l.inst = tlas_refs[k];
        l.blas_root = x.blas_root;
        l.flags = x.flags;
        l.pad = 0;
    }
    HIP_TRY(c, upload(c->tlas_leaf, tlas_leaf.data(), tlas_leaf.size() * sizeof(TlasLeaf), s));
    HIP_TRY(c, upload(c->insts, insts.data(), insts.size() * sizeof(DInstance), s));
    HIP_TRY(c, upload(c->triverts, tri_verts.data(), tri_verts.size() * sizeof(DVertex), s));
    HIP_TRY(c, upload(c->mats, mats.data(), mats.size() * sizeof(DMaterial), s));
    {
        /* a copy of each instance's material next to the instance index (no instance-to-material hop) */
        std::vector<DMaterial> inst_mats(insts.size());
        for (size_t k = 0; k < insts.size(); ++k) inst_mats[k] = mats[insts[k].material];
        HIP_TRY(c, upload(c->instmats, inst_mats.data(), inst_mats.size() * sizeof(DMaterial), s));
    }
    HIP_TRY(c, upload(c->texs, texs.data(), texs.size() * sizeof(DTexture), s));
    HIP_TRY(c, upload(c->tex8, tex8.data(), tex8.size() * sizeof(uint32_t), s));
    HIP_TRY(c, upload(c->texf, texf.data(), texf.size() * sizeof(float4), s));
    HIP_TRY(c, upload(c->lights, lights.data(), lights.size() * sizeof(DLight), s));
    HIP_TRY(c, upload(c->cube, cube.data(), cube.size() * sizeof(float4), s));
    if (cube_w > 0 && (D->environment.type == VVPT_ENV_HDRI || D->environment.type == VVPT_ENV_SOLID_COLOR_WITH_HDRI_LIGHTING)) {
        const std::string err = build_env_importance(c, cube_w);
        if (!err.empty()) return set_err(c, VVPT_DEVICE_LOST, "environment importance grid: " + err);
    }
    c->sh.valid = true;
    c->sh.num_instances = D->num_instances;
    c->sh.num_lights = c->sh.parts[0].num_lights;
    c->sh.scene_flags = (any_transparent ? SCENE_HAS_TRANSPARENT : 0u) | (any_volume_change ? SCENE_HAS_VOLUME_CHANGE : 0u);
    c->sh.walks = any_volume_change;
    for (const DMaterial &m : mats) {
        c->sh.walks = c->sh.walks || (m.flags & 2u);
        for (uint32_t t : {m.tex1[0], m.tex1[1], m.tex1[2], m.tex2[0], m.tex2[1]}) c->sh.textured = c->sh.textured || t >= 3u;
    }
    c->sh.cube_w = cube_w;
    c->sh.cam = D->camera;
    c->sh.env = D->environment;
    c->sh.mats_desc.assign(D->materials, D->materials + D->num_materials);
    return VVPT_OK;
}

vvpt_status vvpt_set_scene(vvpt_ctx *c, const vvpt_scene_desc *D) {
    if (!c || !D) return VVPT_INVALID;
    VVPT_TAKE(c);
    HIP_TRY(c, hipSetDevice(c->device));
    const std::vector<PartRange> parts = {{0u, D->num_instances, 0u, D->num_lights, D->camera, 0u, D->num_materials}};
    return set_scene_parts(c, D, parts);
}

vvpt_status vvpt_set_camera(vvpt_ctx *c, uint32_t scene, const vvpt_camera *camera) {
    if (!c || !camera) return c ? set_err(c, VVPT_INVALID, "no camera") : VVPT_INVALID;
    VVPT_TAKE(c);
    if (!c->sh.valid || scene >= c->sh.parts.size()) return set_err(c, VVPT_INVALID, "no scene with that index");
    if (camera->type != VVPT_CAMERA_PERSPECTIVE && camera->type != VVPT_CAMERA_ORTHOGRAPHIC)
        return set_err(c, VVPT_INVALID, "bad camera type");
    float vi[16];
    if (!inverse4_glm(camera->view, vi)) return set_err(c, VVPT_INVALID, "singular view matrix");
    SceneHost::Part &pt = c->sh.parts[scene];
    pt.cam = *camera;
    if (pt.cam.volume >= 0) pt.cam.volume += (int32_t)pt.mat_begin;
    if (scene == 0) c->sh.cam = pt.cam;
    return VVPT_OK;
}

vvpt_status vvpt_set_scenes(vvpt_ctx *c, const vvpt_scene_desc *scenes, uint32_t count) {
    if (!c || !scenes || count == 0) return c ? set_err(c, VVPT_INVALID, "no scenes") : VVPT_INVALID;
    VVPT_TAKE(c);
    HIP_TRY(c, hipSetDevice(c->device));
    /* merge: meshes, materials, textures and instances concatenated with their indices shifted; each scene is
     * one part; the environment (and its texture) of scene 0 serves every part */
    std::vector<vvpt_mesh> meshes;
    std::vector<vvpt_material> mats;
    std::vector<vvpt_texture> texs;
    std::vector<vvpt_instance> insts;
    std::vector<vvpt_light> lights;
    std::vector<PartRange> parts;
    for (uint32_t k = 0; k < count; ++k) {
        const vvpt_scene_desc &D = scenes[k];
        const uint32_t mo = (uint32_t)meshes.size(), ma = (uint32_t)mats.size(), to = (uint32_t)texs.size();
        for (uint32_t i = 0; i < D.num_instances; ++i)
            if (D.instances[i].mesh >= D.num_meshes || D.instances[i].material >= D.num_materials)
                return set_err(c, VVPT_INVALID, "instance references a missing mesh or material");
        meshes.insert(meshes.end(), D.meshes, D.meshes + D.num_meshes);
        texs.insert(texs.end(), D.textures, D.textures + D.num_textures);
        for (uint32_t i = 0; i < D.num_materials; ++i) {
            vvpt_material m = D.materials[i];
            int32_t *ids[7] = {&m.tex_albedo, &m.tex_metallic, &m.tex_roughness, &m.tex_ao, &m.tex_emissive,
                               &m.tex_normal, &m.tex_alpha};
            for (int32_t *id : ids)
                if (*id >= 0) *id = ((uint32_t)*id < D.num_textures) ? *id + (int32_t)to : -1;
            mats.push_back(m);
        }
        PartRange pr;
        pr.inst_begin = (uint32_t)insts.size();
        pr.inst_count = D.num_instances;
        pr.light_begin = (uint32_t)lights.size();
        pr.light_count = D.num_lights;
        pr.cam = D.camera;
        if (pr.cam.volume >= 0) pr.cam.volume += (int32_t)ma;
        pr.mat_begin = ma;
        pr.mat_count = D.num_materials;
        for (uint32_t i = 0; i < D.num_instances; ++i) {
            vvpt_instance x = D.instances[i];
            x.mesh += mo;
            x.material += ma;
            if (x.front_volume >= 0) x.front_volume += (int32_t)ma;
            if (x.back_volume >= 0) x.back_volume += (int32_t)ma;
            insts.push_back(x);
        }
        lights.insert(lights.end(), D.lights, D.lights + D.num_lights);
        parts.push_back(pr);
    }
    vvpt_scene_desc M = scenes[0];
    M.meshes = meshes.data();
    M.num_meshes = (uint32_t)meshes.size();
    M.materials = mats.data();
    M.num_materials = (uint32_t)mats.size();
    M.textures = texs.data();
    M.num_textures = (uint32_t)texs.size();
    M.instances = insts.data();
    M.num_instances = (uint32_t)insts.size();
    M.lights = lights.data();
    M.num_lights = (uint32_t)lights.size();
    return set_scene_parts(c, &M, parts);
}

vvpt_status vvpt_get_bvh_info(const vvpt_ctx *c, vvpt_bvh_info *out) {
    if (!c || !out || !c->sh.valid) return VVPT_INVALID;
    out->tlas_nodes = c->sh.tlas_nodes;
    out->blas_nodes = c->sh.blas_nodes;
    out->triangles = c->sh.num_triangles;
    out->instances = c->sh.num_instances;
    out->max_depth = c->sh.max_depth;
    out->node_bytes = sizeof(WideNode);
    out->triangle_bytes = sizeof(LeafTri);
    return VVPT_OK;
}

vvpt_status vvpt_sample_sequence(vvpt_ctx *c, uint32_t pixel, uint32_t seed, uint32_t first, uint32_t count,
                                 uint32_t dims, float *out) {
    if (!out || (uint64_t)count * dims > (1ull << 28)) return c ? set_err(c, VVPT_INVALID, "invalid sampler request") : VVPT_INVALID;
    const uint32_t key = sampler_key(pixel, seed);
    const size_t n = (size_t)count * dims;
    if (!c) {
        for (size_t i = 0; i < n; ++i) out[i] = sampler_float(key, first + (uint32_t)(i / dims), (uint32_t)(i % dims));
        return VVPT_OK;
    }
    if (n == 0) return VVPT_OK;
    VVPT_TAKE(c);
    HIP_TRY(c, hipSetDevice(c->device));
    DevBuf buf;
    HIP_TRY(c, ensure(buf, n * sizeof(float)));
    hipLaunchKernelGGL(k_sample_sequence, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, c->stream, key, first, count,
                       dims, (float *)buf.p);
    hipError_t e = hipGetLastError();
    if (e == hipSuccess) e = hipMemcpyAsync(out, buf.p, n * sizeof(float), hipMemcpyDeviceToHost, c->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(c->stream);
    release(buf);
    if (e != hipSuccess) return set_err(c, VVPT_DEVICE_LOST, std::string("sampler: ") + hipGetErrorString(e));
    return VVPT_OK;
}

/* ------------------------------------------------------------ NRC hooks -- */

/* The caller has taken the context. */
/* The cache's schedule from the context's options: finest grid resolution and Adam learning rate. */
static void nrc_apply_options(vvpt_ctx *c) {
    c->nrc->set_max_resolution(c->opt.nrc_max_resolution > 0.0f ? c->opt.nrc_max_resolution : kNrcMaxRes);
    c->nrc->lr0 = c->opt.nrc_learning_rate > 0.0f ? c->opt.nrc_learning_rate : 3e-3f;
}

static vvpt_status nrc_ready(vvpt_ctx *c) {
    HIP_TRY(c, hipSetDevice(c->device));
    if (!c->nrc) {
        c->nrc = new NrcModel();
        const std::string e = c->nrc->init(c->stream, 1u);
        if (!e.empty()) return set_err(c, VVPT_OOM, "NRC init: " + e);
        nrc_apply_options(c);
    }
    c->nrc->stream = c->stream;
    return VVPT_OK;
}

vvpt_status vvpt_nrc_reset(vvpt_ctx *c, uint32_t seed, const float *lo, const float *hi) {
    if (!c) return VVPT_INVALID;
    VVPT_TAKE(c);
    vvpt_status st = nrc_ready(c);
    if (st != VVPT_OK) return st;
    const std::string e = c->nrc->init(c->stream, seed);
    if (!e.empty()) return set_err(c, VVPT_DEVICE_LOST, "NRC init: " + e);
    if (lo && hi) c->nrc->set_bounds(lo, hi);
    nrc_apply_options(c);
    return VVPT_OK;
}

vvpt_status vvpt_nrc_infer(vvpt_ctx *c, const float *inputs, uint32_t n, float *out) {
    if (!c) return VVPT_INVALID;
    VVPT_TAKE(c);
    vvpt_status st = nrc_ready(c);
    if (st != VVPT_OK) return st;
    if (!inputs || !out || n > NrcModel::kMaxBatch) return set_err(c, VVPT_INVALID, "NRC batch out of range");
    NrcModel &M = *c->nrc;
    HIP_TRY(c, hipMemcpyAsync(M.in, inputs, (size_t)n * kNrcIn * sizeof(float), hipMemcpyHostToDevice, c->stream));
    const std::string e = M.infer((const float *)M.in, n, (float *)M.pred);
    if (!e.empty()) return set_err(c, VVPT_DEVICE_LOST, "NRC inference: " + e);
    HIP_TRY(c, hipMemcpyAsync(out, M.pred, (size_t)n * 3 * sizeof(float), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    return VVPT_OK;
}

vvpt_status vvpt_nrc_train(vvpt_ctx *c, const float *inputs, const float *targets, uint32_t n, uint32_t steps,
                           float *losses) {
    if (!c) return VVPT_INVALID;
    VVPT_TAKE(c);
    vvpt_status st = nrc_ready(c);
    if (st != VVPT_OK) return st;
    if (!inputs || !targets || n == 0 || n > NrcModel::kMaxBatch) return set_err(c, VVPT_INVALID, "NRC batch out of range");
    NrcModel &M = *c->nrc;
    HIP_TRY(c, hipMemcpyAsync(M.in, inputs, (size_t)n * kNrcIn * sizeof(float), hipMemcpyHostToDevice, c->stream));
    HIP_TRY(c, hipMemcpyAsync(M.tgt, targets, (size_t)n * 3 * sizeof(float), hipMemcpyHostToDevice, c->stream));
    for (uint32_t k = 0; k < steps; ++k) {
        const std::string e = M.train_step((const float *)M.in, (const float *)M.tgt, n, losses ? losses + k : nullptr);
        if (!e.empty()) return set_err(c, VVPT_DEVICE_LOST, "NRC training: " + e);
    }
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    return VVPT_OK;
}

vvpt_status vvpt_nrc_gradients(vvpt_ctx *c, const float *inputs, const float *targets, uint32_t n, float *loss,
                               float *mlp_grad, float *grid_grad) {
    if (!c) return VVPT_INVALID;
    VVPT_TAKE(c);
    vvpt_status st = nrc_ready(c);
    if (st != VVPT_OK) return st;
    if (!inputs || !targets || n == 0 || n > NrcModel::kMaxBatch) return set_err(c, VVPT_INVALID, "NRC batch out of range");
    NrcModel &M = *c->nrc;
    HIP_TRY(c, hipMemcpyAsync(M.in, inputs, (size_t)n * kNrcIn * sizeof(float), hipMemcpyHostToDevice, c->stream));
    HIP_TRY(c, hipMemcpyAsync(M.tgt, targets, (size_t)n * 3 * sizeof(float), hipMemcpyHostToDevice, c->stream));
    const std::string e = M.gradients((const float *)M.in, (const float *)M.tgt, n, loss);
    if (!e.empty()) return set_err(c, VVPT_DEVICE_LOST, "NRC gradients: " + e);
    if (mlp_grad) HIP_TRY(c, hipMemcpyAsync(mlp_grad, M.wg, kNrcMlpParams * sizeof(float), hipMemcpyDeviceToHost, c->stream));
    if (grid_grad) HIP_TRY(c, hipMemcpyAsync(grid_grad, M.gg, kNrcGridParams * sizeof(float), hipMemcpyDeviceToHost, c->stream));
    HIP_TRY(c, hipMemsetAsync(M.wg, 0, kNrcMlpParams * sizeof(float), c->stream));
    HIP_TRY(c, hipMemsetAsync(M.gg, 0, kNrcGridParams * sizeof(float), c->stream));
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    return VVPT_OK;
}

vvpt_status vvpt_nrc_params(vvpt_ctx *c, float *mlp, float *grid, int write) {
    if (!c) return VVPT_INVALID;
    VVPT_TAKE(c);
    vvpt_status st = nrc_ready(c);
    if (st != VVPT_OK) return st;
    NrcModel &M = *c->nrc;
    const hipMemcpyKind k = write ? hipMemcpyHostToDevice : hipMemcpyDeviceToHost;
    if (mlp) HIP_TRY(c, hipMemcpyAsync(write ? M.w32 : (void *)mlp, write ? (const void *)mlp : M.w32,
                                      kNrcMlpParams * sizeof(float), k, c->stream));
    if (grid) HIP_TRY(c, hipMemcpyAsync(write ? M.grid : (void *)grid, write ? (const void *)grid : M.grid,
                                       kNrcGridParams * sizeof(float), k, c->stream));
    HIP_TRY(c, hipStreamSynchronize(c->stream));
    if (write && grid) {
        const std::string e = M.refresh_grid16();
        if (!e.empty()) return set_err(c, VVPT_DEVICE_LOST, "NRC grid: " + e);
        HIP_TRY(c, hipStreamSynchronize(c->stream));
    }
    if (write && mlp) {
        std::vector<uint16_t> h(kNrcMlpParams);
        for (uint32_t i = 0; i < kNrcMlpParams; ++i) h[i] = f32_to_bf16(mlp[i]);
        HIP_TRY(c, hipMemcpy(M.w16, h.data(), h.size() * sizeof(uint16_t), hipMemcpyHostToDevice));
        const std::string e = M.pack_weights();
        if (!e.empty()) return set_err(c, VVPT_DEVICE_LOST, "NRC weights: " + e);
        HIP_TRY(c, hipStreamSynchronize(c->stream));
    }
    return VVPT_OK;
}

vvpt_status vvpt_set_builder(vvpt_ctx *c, uint32_t builder) {
    if (!c) return VVPT_INVALID;
    VVPT_TAKE(c);
    if (builder != VVPT_BUILDER_SAH && builder != VVPT_BUILDER_LBVH) return set_err(c, VVPT_INVALID, "unknown builder");
    c->builder = builder;
    return VVPT_OK;
}

vvpt_status vvpt_build_lbvh(vvpt_ctx *c, const float *boxes, uint32_t n, uint32_t max_leaf, uint32_t *morton,
                            uint32_t *order, uint32_t *inner, void *nodes, uint32_t *leaf_refs, vvpt_lbvh_info *info) {
    if ((n > 0 && !boxes) || max_leaf < 1 || max_leaf > 3) return c ? set_err(c, VVPT_INVALID, "invalid LBVH arguments") : VVPT_INVALID;
    const bool dbg = morton || order || inner;
    LbvhOutput o;
    if (c) {
        VVPT_TAKE(c);
        HIP_TRY(c, hipSetDevice(c->device));
        const std::string err = lbvh_build_device(boxes, n, max_leaf, dbg, c->stream, o);
        if (!err.empty()) return set_err(c, VVPT_DEVICE_LOST, "LBVH build: " + err);
    } else {
        lbvh_build_host(boxes, n, max_leaf, dbg, o);
    }
    if (morton && !o.codes.empty()) std::memcpy(morton, o.codes.data(), 4 * o.codes.size());
    if (order && !o.order.empty()) std::memcpy(order, o.order.data(), 4 * o.order.size());
    if (inner && !o.inner.empty()) std::memcpy(inner, o.inner.data(), 4 * o.inner.size());
    if (nodes) std::memcpy(nodes, o.nodes.data(), sizeof(WideNode) * o.nodes.size());
    if (leaf_refs && !o.leaf_refs.empty()) std::memcpy(leaf_refs, o.leaf_refs.data(), 4 * o.leaf_refs.size());
    if (info) {
        info->num_nodes = (uint32_t)o.nodes.size();
        info->num_leaf_refs = (uint32_t)o.leaf_refs.size();
        info->depth = o.depth;
        info->build_ms = o.ms;
    }
    return VVPT_OK;
}

}  // extern "C"

namespace {

/* SceneData of this render: view inverse and the per-render projection
 * (VulkanRendererPathTracing.cpp:143-198). */
/* Scene-wide part of the device view (every job of a render shares it). */
vvpt_status make_dscene(vvpt_ctx *c, bool ext, DScene &S) {
    const SceneHost &sh = c->sh;
    std::memset(&S, 0, sizeof(S));
    S.nodes = (const WideNode *)c->nodes.p;
    S.tris = (const LeafTri *)c->tris.p;
    S.tlas_leaf = (const TlasLeaf *)c->tlas_leaf.p;
    S.insts = (const DInstance *)c->insts.p;
    S.tri_verts = (const DVertex *)c->triverts.p;
    S.mats = (const DMaterial *)c->mats.p;
    S.inst_mats = (const DMaterial *)c->instmats.p;
    S.texs = (const DTexture *)c->texs.p;
    S.tex8 = (const uint32_t *)c->tex8.p;
    S.texf = (const float4 *)c->texf.p;
    S.lights = (const DLight *)c->lights.p;
    S.cube = (const float4 *)c->cube.p;
    S.srgb_lut = (const float *)c->srgb.p;
    S.cube_w = sh.cube_w;
    S.scene_flags = sh.scene_flags;
    S.env_type = sh.env.type;
    S.bg[0] = sh.env.background[0];
    S.bg[1] = sh.env.background[1];
    S.bg[2] = sh.env.background[2];
    S.env_intensity = sh.env.intensity;
    S.flat_normal[0] = S.flat_normal[1] = 128.0f / 255.0f; /* texel 2: 0xFFFF8080 */
    S.flat_normal[2] = 1.0f;
    if (ext && sh.env_mw > 0) { /* extended mode: the environment becomes one more light to choose */
        S.env_mw = sh.env_mw;
        S.env_mh = sh.env_mh;
        S.env_prob = (const float *)c->env_prob.p;
        S.env_alias = (const uint32_t *)c->env_alias.p;
        S.env_cpdf = (const float *)c->env_cpdf.p;
    }
    return VVPT_OK;
}

/* Per-job part: SceneData of the job's scene part at the job's resolution (VulkanRendererPathTracing.cpp:143-198)
 * and the RenderInfo fields.  Work-item placement (item_begin, items, batch_begin) is set by the caller. */
vvpt_status make_jobview(vvpt_ctx *c, uint32_t part, const vvpt_render_info &info, bool ext, JobView &J) {
    const SceneHost &sh = c->sh;
    if (part >= sh.parts.size()) return set_err(c, VVPT_INVALID, "job references a missing scene");
    const SceneHost::Part &pt = sh.parts[part];
    const uint32_t W = info.width, H = info.height;
    std::memset(&J, 0, sizeof(J));
    J.tlas_root = pt.tlas_root;
    J.light_begin = pt.light_begin;
    J.num_lights = pt.num_lights;
    J.num_sel = pt.num_lights + ((ext && sh.env_mw > 0) ? 1u : 0u);
    J.scene_flags = pt.scene_flags;
    const vvpt_camera &k = pt.cam;
    if (!inverse4_glm(k.view, J.vi)) return set_err(c, VVPT_INVALID, "singular view matrix");
    float pf[16] = {0};
    float n = k.znear, f = k.zfar;
    if (k.type == VVPT_CAMERA_PERSPECTIVE) {
        /* glm::perspective with GLM_FORCE_DEPTH_ZERO_TO_ONE (core/Camera.hpp:5) */
        float fovy = k.fov_degrees * 0.01745329251994329577f;
        float aspect = (float)W / (float)H;
        float th = std::tan(fovy / 2.0f);
        pf[0] = 1.0f / (aspect * th);
        pf[5] = 1.0f / th;
        pf[10] = f / (n - f);
        pf[11] = -1.0f;
        pf[14] = -(f * n) / (f - n);
    } else {
        float l = -(float)W / 2, r = (float)W / 2, b = -(float)H / 2, t = (float)H / 2;
        pf[0] = 2.0f / (r - l);
        pf[5] = 2.0f / (t - b);
        pf[10] = -1.0f / (f - n);
        pf[12] = -(r + l) / (r - l);
        pf[13] = -(t + b) / (t - b);
        pf[14] = -n / (f - n);
        pf[15] = 1.0f;
    }
    pf[5] *= -1.0f; /* VulkanRendererPathTracing.cpp:153 */
    if (!inverse4_glm(pf, J.pi)) return set_err(c, VVPT_INVALID, "singular projection");
    J.lens = k.lens_radius;
    J.focal = k.focal_distance;
    J.znear = k.znear;
    J.zfar = k.zfar;
    J.cam_volume = -1;
    if (k.volume >= 0 && (uint32_t)k.volume < sh.mats_desc.size() && sh.mats_desc[k.volume].type == VVPT_MATERIAL_VOLUME)
        J.cam_volume = k.volume;
    J.W = W;
    J.H = H;
    J.npix = W * H;
    J.batch_size = info.batch_size;
    J.depth = info.depth;
    J.seed = info.seed;
    J.total_samples = (float)(info.batch_size * (info.samples / info.batch_size)); /* :798-799 */
    return VVPT_OK;
}

/* Traversal stacks live in LDS (8 bytes per entry per lane), which bounds the trace kernels' occupancy, so the
 * kernels are compiled for several depths and a render uses the smallest stack that holds max_depth + 2 entries.
 * A walk pushes a node group only on a level that still has siblings to visit (at most depth - 1 entries per
 * BVH) plus the two entries that keep the TLAS position during a BLAS walk: at most max_depth entries. */
constexpr int kStackSizes[] = {10, 12, 16, 24, 32, 64};

int stack_size_for(uint32_t depth) {
    for (int sz : kStackSizes)
        if ((int)depth + 2 <= sz) return sz;
    return 0;
}

/* Calls f(std::integral_constant<int, STACK>) for the compiled stack size STACK. */
template <class F>
bool with_stack(int stack, F &&f) {
    switch (stack) {
        case 10: f(std::integral_constant<int, 10>()); return true;
        case 12: f(std::integral_constant<int, 12>()); return true;
        case 16: f(std::integral_constant<int, 16>()); return true;
        case 24: f(std::integral_constant<int, 24>()); return true;
        case 32: f(std::integral_constant<int, 32>()); return true;
        case 64: f(std::integral_constant<int, 64>()); return true;
        default: return false;
    }
}

template <int STACK, bool MULTI>
void launch_extend(bool count, dim3 g, hipStream_t s, const DScene &S, const RenderParams &P, const PathState &st,
                   uint32_t cur) {
    if (count)
        hipLaunchKernelGGL((k_extend<STACK, true, MULTI>), g, dim3(kTraceBlock), 0, s, S, P, st, cur);
    else
        hipLaunchKernelGGL((k_extend<STACK, false, MULTI>), g, dim3(kTraceBlock), 0, s, S, P, st, cur);
}
template <int STACK, bool MULTI>
void launch_shadow(bool count, bool alpha, dim3 g, hipStream_t s, const DScene &S, const RenderParams &P,
                   const PathState &st) {
    if (alpha) {
        if (count)
            hipLaunchKernelGGL((k_shadow<STACK, true, true, MULTI>), g, dim3(kTraceBlock), 0, s, S, P, st);
        else
            hipLaunchKernelGGL((k_shadow<STACK, false, true, MULTI>), g, dim3(kTraceBlock), 0, s, S, P, st);
    } else {
        if (count)
            hipLaunchKernelGGL((k_shadow<STACK, true, false, MULTI>), g, dim3(kTraceBlock), 0, s, S, P, st);
        else
            hipLaunchKernelGGL((k_shadow<STACK, false, false, MULTI>), g, dim3(kTraceBlock), 0, s, S, P, st);
    }
}
template <int STACK, bool MULTI>
void launch_secondary(bool count, dim3 g, hipStream_t s, const DScene &S, const RenderParams &P, const PathState &st) {
    if (count)
        hipLaunchKernelGGL((k_secondary<STACK, true, MULTI>), g, dim3(kTraceBlock), 0, s, S, P, st);
    else
        hipLaunchKernelGGL((k_secondary<STACK, false, MULTI>), g, dim3(kTraceBlock), 0, s, S, P, st);
}

/* The features a render's k_shade is compiled for (kernels.h Features). */
struct RenderFeatures {
    bool ext, nrc, tex, vol;
};
/* Calls f(Features<...>()) for the compiled features that cover fx.  A batched render has no radiance cache and always
 * runs the code with media, whatever its jobs: most batches hold a job in one, and the batched variant without media is
 * the one whose first launch through a captured graph ended in a memory fault whose cause is not shown. */
template <bool MULTI, class F>
void with_features(const RenderFeatures &fx, F &&f) {
    using T = std::true_type;
    using N = std::false_type;
    auto tv = [&](auto e, auto n) {
        constexpr bool E = decltype(e)::value, N_ = decltype(n)::value;
        if constexpr (MULTI) {
            if (fx.tex) f(Features<E, N_, true, true>());
            else f(Features<E, N_, false, true>());
        } else {
            if (fx.tex && fx.vol) f(Features<E, N_, true, true>());
            else if (fx.tex) f(Features<E, N_, true, false>());
            else if (fx.vol) f(Features<E, N_, false, true>());
            else f(Features<E, N_, false, false>());
        }
    };
    if constexpr (!MULTI) {
        if (fx.nrc) {
            tv(T(), T());
            return;
        }
    }
    if (fx.ext) tv(T(), N());
    else tv(N(), N());
}

/* Per-launch hipEvent pairs; launches of kernel k are bracketed by events 2i, 2i+1. */
struct KernelTimer {
    vvpt_ctx *c;
    bool on;
    hipStream_t s;
    std::vector<int> kind;
    size_t used = 0;
    hipError_t begin(int k) {
        if (!on) return hipSuccess;
        if (c->kev.size() < used + 2) {
            for (int i = 0; i < 2; ++i) {
                hipEvent_t e;
                hipError_t r = hipEventCreate(&e);
                if (r != hipSuccess) return r;
                c->kev.push_back(e);
            }
        }
        kind.push_back(k);
        return hipEventRecord(c->kev[used++], s);
    }
    hipError_t end() { return on ? hipEventRecord(c->kev[used++], s) : hipSuccess; }
    hipError_t collect(vvpt_stats *st) {
        for (size_t i = 0; i < kind.size(); ++i) {
            float ms = 0.0f;
            hipError_t r = hipEventElapsedTime(&ms, c->kev[2 * i], c->kev[2 * i + 1]);
            if (r != hipSuccess) return r;
            st->kernel_ms[kind[i]] += ms;
            st->kernel_launches[kind[i]] += 1;
        }
        return hipSuccess;
    }
};

/* One job of a render: its scene part, RenderInfo and device outputs. */
struct JobSpec {
    uint32_t part;
    vvpt_render_info info;
    float *rad, *alb, *nrm;
};

/* Items per chunk of a batched render's item order (chunks are dealt round-robin over the item shards). */
constexpr uint32_t kItemChunk = 4096;

/* Training paths of the radiance cache's first frame, in units of the later frames' (the first training round
 * starts from the untrained cache and decides what the second frame's queries return). */
constexpr double kNrcFirstFrameScale = 2.0;

/* Body of vvpt_render_device (one job, MULTI = false: launch windows of batches, AOVs, the radiance cache) and of
 * vvpt_render_jobs (MULTI = true: every job's work items in one window, shortest job first, completion times). */
vvpt_status render_core(vvpt_ctx *c, const std::vector<JobSpec> &jobs, bool multi, uint32_t flags, hipStream_t s,
                        vvpt_stats *stats, double *done_ms) {
    const bool count_nodes = (flags & VVPT_FLAG_COUNT_NODES) != 0u;
    const bool nrc_flag = !multi && (flags & VVPT_FLAG_NRC) != 0u;
    const bool ext = nrc_flag || (flags & VVPT_FLAG_EXTENDED) != 0u;
    const bool aovs = !multi && (flags & VVPT_FLAG_AOVS) != 0u;
    const bool timing = (flags & VVPT_FLAG_KERNEL_TIMING) != 0u && stats != nullptr;
    const bool graph = (flags & VVPT_FLAG_GRAPH) != 0u;
    if (graph && (nrc_flag || timing))
        return set_err(c, VVPT_INVALID, "VVPT_FLAG_GRAPH excludes VVPT_FLAG_NRC and VVPT_FLAG_KERNEL_TIMING");
    DScene S;
    vvpt_status st0 = make_dscene(c, ext, S);
    if (st0 != VVPT_OK) return st0;
    const size_t njobs = jobs.size();
    std::vector<JobView> J(njobs);
    std::vector<uint32_t> batches(njobs);
    for (size_t i = 0; i < njobs; ++i) {
        st0 = make_jobview(c, jobs[i].part, jobs[i].info, ext, J[i]);
        if (st0 != VVPT_OK) return st0;
        batches[i] = jobs[i].info.samples / jobs[i].info.batch_size; /* remainder dropped (:798-799) */
    }
    const int STACK = stack_size_for(c->sh.max_depth);
    if (STACK == 0) return set_err(c, VVPT_UNSUPPORTED, "BVH too deep for the traversal stack");

    /* the cache trains between frames of nrc_frame_batches batches (default 4); a render of one frame never
     * queries it (the first frame only trains, and no training follows the last), so it runs as the extended
     * estimator without recording training paths */
    const uint32_t frame_batches = c->opt.nrc_frame_batches ? c->opt.nrc_frame_batches : 4u;
    const bool nrc = nrc_flag && batches[0] > frame_batches;
    /* Launch windows.  A single render covers `win` batches per window (the per-batch partial results bound the
     * memory); a batched render places every job's work items in one window, cheapest job first. */
    const vvpt_options &opt = c->opt;
    const size_t max_part_bytes = opt.max_partial_bytes ? (size_t)opt.max_partial_bytes : ((size_t)(multi ? 32 : 8) << 30);
    uint64_t total_items = 0;
    uint32_t win = 1, items_max = 0;
    double nrc_paths = 0.0; /* radiance cache: training paths per frame */
    std::vector<JobView> djobs; /* batched: the jobs with work items, in item order */
    std::vector<int64_t> dindex(njobs, -1);
    if (!multi) {
        const uint32_t npix = J[0].npix;
        const size_t per_batch = (size_t)npix * sizeof(float4) * (aovs ? 3 : 1);
        win = (uint32_t)std::max<size_t>(1, std::min<size_t>(batches[0], max_part_bytes / per_batch));
        if (nrc) win = std::min(win, frame_batches);
        items_max = win * npix;
        total_items = (uint64_t)batches[0] * npix;
    } else {
        std::vector<uint32_t> order(njobs);
        for (size_t i = 0; i < njobs; ++i) order[i] = (uint32_t)i;
        auto cost = [&](uint32_t i) { return (double)J[i].npix * batches[i] * J[i].batch_size * J[i].depth; };
        std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) { return cost(a) < cost(b); });
        for (uint32_t i : order) {
            const uint64_t n = (uint64_t)J[i].npix * batches[i];
            if (n == 0) continue;
            if (total_items + n > 0xffff0000ull) return set_err(c, VVPT_UNSUPPORTED, "batch holds 2^32 or more work items");
            J[i].item_begin = (uint32_t)total_items;
            J[i].items = (uint32_t)n;
            dindex[i] = (int64_t)djobs.size();
            djobs.push_back(J[i]);
            total_items += n;
        }
        if (total_items * sizeof(float4) > max_part_bytes)
            return set_err(c, VVPT_UNSUPPORTED, "batch needs more partial-result memory than VVPT_MAX_PARTIAL_BYTES");
        items_max = (uint32_t)total_items;
    }
    /* k_resolve writes the image of a job with work (its first window stores, later windows add); a job with no
     * complete batch gets zeros */
    for (size_t i = 0; i < njobs; ++i) {
        if (batches[i] == 0u) {
            const size_t np = (size_t)J[i].npix * 16;
            HIP_TRY(c, hipMemsetAsync(jobs[i].rad, 0, np, s));
            if (aovs) {
                HIP_TRY(c, hipMemsetAsync(jobs[i].alb, 0, np, s));
                HIP_TRY(c, hipMemsetAsync(jobs[i].nrm, 0, np, s));
            }
        }
        if (done_ms) done_ms[i] = 0.0;
    }
    if (total_items == 0) {
        if (stats) std::memset(stats, 0, sizeof(*stats));
        HIP_TRY(c, hipStreamSynchronize(s));
        return VVPT_OK;
    }
    /* Path slots (about 460 B each): a trace launch ends with a tail in which lanes run out of rays, so the more
     * rays a launch holds per lane the smaller that tail; 2^25 slots (15 GB) keep every work item of a 1080p,
     * 16-batch render in flight at once (measured on the 1080p icosphere field with 12 trace and 16 shade blocks
     * per CU: 2^22 slots 621, 2^23 660, 2^24 681, 2^25 699 Msamples/s; the block counts move it by 1 %).
     * vvpt_autotune may pick another count. */
    uint32_t nslots = c->tune.slots;
    nslots = std::max(64u, std::min(nslots, items_max));

    /* path state */
    const size_t N = nslots;
    const size_t sizes[] = {
        4, 4, 4, 4, 4,                              /* item rng ctr vol flags */
        16, 16, 16, 16, 16, 16, 16, 16, 16, 16,      /* orig dir beta nee L accR accA accN payA payN */
        64,                                         /* hit (one 64-byte record per slot) */
        48, 48, 48, 12,                             /* sec_o sec_d sec_c sec_v (3 per slot, planar) */
        4, 8, 4                                     /* nrct spread job */
    };
    constexpr int NF = sizeof(sizes) / sizeof(sizes[0]);
    size_t offs[NF], total = 0;
    for (int i = 0; i < NF; ++i) {
        offs[i] = total;
        total += ((sizes[i] * N + 255) / 256) * 256;
    }
    HIP_TRY(c, ensure(c->state, total));
    /* A shard receives the output of at most ceil(N / (64 kShards)) input waves, each appending at most 64 entries
     * per record kind: cap1 entries per shard hold one record per slot.  The secondary queue holds three records
     * per slot and the shadow queue two (a slot's light-sample segment and the 1 - alpha product in front of the
     * emitter its previous bounce found through a transparent surface can both be queued in one iteration). */
    const uint32_t cap1 = queue_shard_capacity(N);
    HIP_TRY(c, ensure(c->queues, (size_t)kShards * cap1 * kQueueBlocks * sizeof(uint32_t)));
    HIP_TRY(c, ensure(c->counters, kCounterBytes));
    HIP_TRY(c, ensure(c->stats, (size_t)kShards * kStatStride * sizeof(unsigned long long)));
    HIP_TRY(c, ensure(c->partials, (size_t)items_max * sizeof(float4) * (aovs ? 3 : 1)));
    char *sb = (char *)c->state.p;
    PathState st;
    int f = 0;
    st.item = (uint32_t *)(sb + offs[f++]);
    st.rng = (uint32_t *)(sb + offs[f++]);
    st.ctr = (uint32_t *)(sb + offs[f++]);
    st.vol = (uint32_t *)(sb + offs[f++]);
    st.flags = (uint32_t *)(sb + offs[f++]);
    st.orig = (float4 *)(sb + offs[f++]);
    st.dir = (float4 *)(sb + offs[f++]);
    st.beta = (float4 *)(sb + offs[f++]);
    st.nee = (float4 *)(sb + offs[f++]);
    st.L = (float4 *)(sb + offs[f++]);
    st.accR = (float4 *)(sb + offs[f++]);
    st.accA = (float4 *)(sb + offs[f++]);
    st.accN = (float4 *)(sb + offs[f++]);
    st.payA = (float4 *)(sb + offs[f++]);
    st.payN = (float4 *)(sb + offs[f++]);
    st.hit = (float4 *)(sb + offs[f++]);
    st.sec_o = (float4 *)(sb + offs[f++]);
    st.sec_d = (float4 *)(sb + offs[f++]);
    st.sec_c = (float4 *)(sb + offs[f++]);
    st.sec_v = (uint32_t *)(sb + offs[f++]);
    st.nsec = nslots;
    st.nrct = (uint32_t *)(sb + offs[f++]);
    st.spread = (float2 *)(sb + offs[f++]);
    st.job = (uint32_t *)(sb + offs[f++]);

    RenderParams P;
    std::memset(&P, 0, sizeof(P));
    P.aovs = aovs ? 1u : 0u;
    uint32_t *q = (uint32_t *)c->queues.p;
    uint32_t *cb = (uint32_t *)c->counters.p;
    auto mkq = [&](uint32_t *data, uint32_t cap, uint32_t slot) {
        SQueue x;
        x.data = data;
        x.cap = cap;
        x.count = cb + (size_t)slot * kShards * kPad;
        x.fetch = cb + (size_t)(slot + 1) * kShards * kPad;
        return x;
    };
    P.ext[0] = mkq(q, kExtendRecords * cap1, CB_EXT0);
    P.ext[1] = mkq(q + (size_t)kShards * cap1, kExtendRecords * cap1, CB_EXT1);
    P.sec = mkq(q + (size_t)2 * kShards * cap1, kSecondaryRecords * cap1, CB_SEC);
    P.shd = mkq(q + (size_t)(2 + kSecondaryRecords) * kShards * cap1, kShadowRecords * cap1, CB_SHD);
    if (nrc) {
        /* radiance cache: training blocks of up to min(depth, 16) vertices, 65536 training samples per frame,
         * one query slot per path slot */
        const vvpt_render_info &info = jobs[0].info;
        if (!c->nrc) c->nrc = new NrcModel();
        std::string e = c->nrc->init(s, info.seed * 2654435761u + 17u);
        if (!e.empty()) return set_err(c, VVPT_OOM, "NRC: " + e);
        c->nrc->set_bounds(c->sh.scene_lo, c->sh.scene_hi);
        nrc_apply_options(c);
        /* The fallback: queries only where the cache's error estimate (from the training samples, predicted before
         * they were trained on) is within tolerance; elsewhere the path continues in the plain estimator.  Off for
         * the untrained control, whose cache never sees a training sample. */
        if (opt.nrc_tolerance >= 0.0f && !(flags & VVPT_FLAG_NRC_UNTRAINED)) {
            P.nrc_ok = (const uint8_t *)c->nrc->ok;
            for (int a = 0; a < 3; ++a) {
                const float ext = c->sh.scene_hi[a] - c->sh.scene_lo[a];
                P.nrc_lo[a] = c->sh.scene_lo[a];
                P.nrc_cells[a] = ext > 0.0f ? (float)kNrcErrRes / ext : 0.0f;
            }
        }
        P.nrc = 1u;
        P.nrc_vmax = std::min<uint32_t>(info.depth, 16u);
        /* Training paths per frame: 0.042 per pixel, between 22,000 (the published real-time setting, ~65,536
         * recorded vertices) and 88,000 (~260,000 vertices at 1080p); one Adam step per 16,384 vertices.  Measured
         * on the Cornell box at 1080p against its 65,536-spp render (learning rate 0.003, finest grid 128): RMSE at
         * 64 / 256 spp and bias 0.00448 / 0.00179 / 0.0006 with 66,000 paths, 0.00437 / 0.00173 / 0.0008 with
         * 88,000, 0.00443 / 0.00180 / 0.0010 with 110,000, 0.00409 / 0.00225 / 0.0016 with 176,000 (sooner to
         * RMSE 4e-3, behind the extended estimator's 0.00208 at 256 spp); on a 480x270 field 88,000 paths raised
         * the frame-mean bias from below 1 % to 3 %, so small frames keep 22,000;
         * more epochs over fewer paths overfit the noisy targets; Adam batches of 16,384 beat 8,192 (unstable) and
         * 32,768 / 65,536 (too few steps per frame: biased).  vvpt_options overrides the training volume, epochs,
         * termination constant and Adam batch. */
        /* room for every vertex of the first frame's training paths: with more records than room, the first ones
         * recorded (those of the shortest paths, which finish first) would be the ones trained on */
        P.nrc_tcap = opt.nrc_train_cap ? std::max(16384u, opt.nrc_train_cap) : 524288u;
        P.nrc_c = opt.nrc_spread > 0.0f ? opt.nrc_spread : 0.01f;
        double paths = opt.nrc_paths ? (double)opt.nrc_paths : std::min(88000.0, std::max(22000.0, 0.042 * J[0].npix));
        nrc_paths = paths;
        const double frac = std::min(1.0, paths / ((double)J[0].npix * info.batch_size * win));
        P.nrc_blocks = std::max(32768u, (uint32_t)(kNrcFirstFrameScale * paths * 1.5));
        P.nrc_thresh = (uint32_t)std::min(4294967295.0, frac * 4294967296.0);
        const size_t pool = (size_t)P.nrc_blocks * P.nrc_vmax * 16 * sizeof(float);
        const size_t tin = (size_t)P.nrc_tcap * 10 * sizeof(float), ttgt = (size_t)P.nrc_tcap * 3 * sizeof(float);
        const size_t qin = (size_t)N * 10 * sizeof(float), qslot = (size_t)N * sizeof(uint32_t),
                     qpred = (size_t)N * 3 * sizeof(float);
        HIP_TRY(c, ensure(c->nrcbuf, 256 + pool + tin + ttgt + qin + qslot + qpred + 6 * 256));
        char *nb = (char *)c->nrcbuf.p;
        auto take = [&](size_t bytes) {
            char *r = nb;
            nb += (bytes + 255) / 256 * 256;
            return r;
        };
        P.nrc_ctr = (uint32_t *)take(256);
        P.nrc_pool = (float *)take(pool);
        P.nrc_tin = (float *)take(tin);
        P.nrc_ttgt = (float *)take(ttgt);
        P.nrc_qin = (float *)take(qin);
        P.nrc_qslot = (uint32_t *)take(qslot);
        P.nrc_qpred = (float *)take(qpred);
        const std::string re = c->nrc->reserve_queries(nslots); /* the queries' grid features */
        if (!re.empty()) return set_err(c, VVPT_OOM, "NRC: " + re);
        P.nrcq = mkq(q + (size_t)(2 + kSecondaryRecords + kShadowRecords) * kShards * cap1, kQueryRecords * cap1, CB_NRCQ);
    }
    P.items = cb + (size_t)CB_ITEMS * kShards * kPad;
    P.stats = (unsigned long long *)c->stats.p;
    float4 *pp = (float4 *)c->partials.p;
    P.partR = pp;
    P.partA = aovs ? pp + items_max : nullptr;
    P.partN = aovs ? pp + 2 * (size_t)items_max : nullptr;

    /* batched: job table, then the jobs' completion ticks (+ the start tick), then their remaining item counts */
    std::vector<char> jobs_host;
    unsigned long long *d_ticks = nullptr;
    if (multi) {
        const size_t nj = djobs.size();
        const size_t jv = (nj * sizeof(JobView) + 255) / 256 * 256, tk = ((nj + 1) * 8 + 255) / 256 * 256;
        HIP_TRY(c, ensure(c->jobbuf, jv + tk + nj * 4));
        char *jb = (char *)c->jobbuf.p;
        d_ticks = (unsigned long long *)(jb + jv);
        uint32_t *d_rem = (uint32_t *)(jb + jv + tk);
        jobs_host.assign(jv + tk + nj * 4, 0);
        for (size_t k = 0; k < nj; ++k) {
            djobs[k].remaining = d_rem + k;
            djobs[k].done_ticks = d_ticks + k;
            const uint32_t items = djobs[k].items;
            std::memcpy(jobs_host.data() + jv + tk + k * 4, &items, 4);
        }
        std::memcpy(jobs_host.data(), djobs.data(), nj * sizeof(JobView));
        HIP_TRY(c, hipMemcpyAsync(jb, jobs_host.data(), jobs_host.size(), hipMemcpyHostToDevice, s));
        S.jobs = (const JobView *)jb;
        S.njobs = (uint32_t)nj;
    }

    HIP_TRY(c, hipMemsetAsync(c->stats.p, 0, (size_t)kShards * kStatStride * sizeof(unsigned long long), s));
    HIP_TRY(c, hipEventRecord(c->ev0, s));

    /* Iteration bound of a launch window (the reference's per-batch fence timeout, :869-876).  A sample lasts at
     * most depth + 2 iterations (one per bounce, a transparent pass-through or a scattering event included, the walk
     * of its last emitter lookup, and one more when it ends with results pending), so a work item needs at most
     * batch_size (depth + 2) slot-iterations.  While items remain unstarted every slot is busy (k_shade refills a slot
     * in the iteration its item ends), so a window of total work T slot-iterations on n slots ends within T / n + one
     * item's length; twice that is the bound.  vvpt_options.max_iterations replaces it as it is. */
    auto window_bound = [&](uint32_t nb_window) -> uint64_t {
        if (opt.max_iterations) return opt.max_iterations;
        double work = 0.0, tail = 0.0;
        if (multi) {
            for (size_t i = 0; i < njobs; ++i) {
                const double per_item = (double)J[i].batch_size * (J[i].depth + 2u);
                work += (double)J[i].npix * batches[i] * per_item;
                if (batches[i]) tail = std::max(tail, per_item);
            }
        } else {
            tail = (double)J[0].batch_size * (J[0].depth + 2u);
            work = (double)J[0].npix * nb_window * tail;
        }
        const double n = (double)std::max<uint32_t>(1u, std::min<uint64_t>(nslots, multi ? items_max : (uint64_t)nb_window * J[0].npix));
        return (uint64_t)(2.0 * (std::ceil(work / n) + tail)) + 8u;
    };

    const uint32_t cus = c->cus;
    uint64_t iterations = 0;
    KernelTimer kt{c, timing, s};
    uint64_t items_done_before = 0;
    uint64_t nrc_trained = 0;
    c->progress.store(0.0f);
    const bool alpha = (S.scene_flags & SCENE_HAS_TRANSPARENT) != 0u;
    /* k_shade queues general walks only for surfaces that change volume or are transparent */
    const bool walks = c->sh.walks;
    RenderFeatures fx = {ext, nrc, c->sh.textured, multi || (S.scene_flags & SCENE_HAS_VOLUME_CHANGE) != 0u};
    for (const JobView &j : J) fx.vol = fx.vol || j.cam_volume >= 0;
    P.media = fx.vol ? 1u : 0u;
    /* launch windows: a batched render has one; a single render covers `win` batches per window */
    std::vector<uint32_t> wins;
    if (multi)
        wins.push_back(0u);
    else
        for (uint32_t b = 0; b < batches[0]; b += win) wins.push_back(std::min(win, batches[0] - b));
    uint32_t b0_next = 0;
    for (size_t w = 0; w < wins.size(); ++w) {
        const uint32_t b0 = b0_next;
        const uint32_t nb = wins[w];
        b0_next += nb;
        if (nrc) { /* the training fraction gives about `paths` training paths in this frame (the first: more) */
            const double paths_w = nrc_paths * (w == 0 ? kNrcFirstFrameScale : 1.0);
            const double frac = std::min(1.0, paths_w / ((double)J[0].npix * jobs[0].info.batch_size * nb));
            P.nrc_thresh = (uint32_t)std::min(4294967295.0, frac * 4294967296.0);
        }
        if (!multi) {
            S.job = J[0];
            S.job.batch_begin = b0;
            S.job.item_begin = 0;
            S.job.items = nb * J[0].npix;
        }
        P.items_total = multi ? items_max : S.job.items;
        P.nslots = std::min<uint32_t>(nslots, P.items_total);
        P.item_chunk = multi ? kItemChunk : 0u;
        P.items_per_shard = multi ? item_shard_size(P.items_total, 0u, P.item_chunk, 0u)
                                  : (P.items_total + kShards - 1) / kShards;
        /* every counter zero; item shard s starts at per - size_s (queue.h item_fetch) */
        std::vector<uint32_t> init(kCounterBytes / 4, 0u);
        for (uint32_t sh = 0; sh < kShards; ++sh)
            init[(size_t)CB_ITEMS * kShards * kPad + sh * kPad] =
                P.items_per_shard - item_shard_size(P.items_total, P.items_per_shard, P.item_chunk, sh);
        HIP_TRY(c, hipMemcpyAsync(cb, init.data(), kCounterBytes, hipMemcpyHostToDevice, s));
        if (nrc) {
            HIP_TRY(c, hipMemsetAsync(P.nrc_ctr, 0, 256, s));
            P.nrc_use = b0 > 0 ? 1u : 0u; /* the first frame only trains */
            /* the last frame's training samples would never be trained on: none are recorded, so every path of
             * that frame may query; a render of a single frame is then the extended estimator itself */
            const bool last = w + 1 == wins.size();
            if (last) P.nrc_thresh = 0u;
            P.nrc = (P.nrc_use || !last) ? 1u : 0u;
        }
        HIP_TRY(c, hipStreamSynchronize(s));
        if (multi) hipLaunchKernelGGL(k_clock_stamp, dim3(1), dim3(64), 0, s, d_ticks + djobs.size());
        /* Slots that can still hold a path: all of them at first, then what the last counter readback found (a slot
         * without a work item never gets one again, so the count only falls).  Launches are sized to it: a lane per
         * ray, up to the tuned block counts.  A trace block without a ray still takes queue counters from the others
         * (same-address atomics) and scans all shards before it ends. */
        uint32_t live = P.nslots;
        dim3 trace_grid, g_shade;
        auto size_grids = [&]() {
            trace_grid = dim3(std::min<uint32_t>((live + kTraceBlock - 1) / kTraceBlock, cus * c->tune.trace_blocks_per_cu));
            g_shade = dim3(std::min<uint32_t>((live + kBlock - 1) / kBlock, cus * c->tune.shade_blocks_per_cu));
        };
        size_grids();

        /* one wavefront iteration: the walks of the previous bounce's secondary records, extend, shade (+ cache
         * queries).  The general walk serves volume boundaries and transparent surfaces only. */
        auto iteration = [&](auto mt, uint32_t cur) -> vvpt_status {
            constexpr bool M = decltype(mt)::value;
            if (walks) {
                HIP_TRY(c, kt.begin(VVPT_K_SECONDARY));
                with_stack(STACK, [&](auto k) { launch_secondary<decltype(k)::value, M>(count_nodes, trace_grid, s, S, P, st); });
                HIP_TRY(c, kt.end());
            }
            HIP_TRY(c, kt.begin(VVPT_K_SHADOW));
            with_stack(STACK, [&](auto k) { launch_shadow<decltype(k)::value, M>(count_nodes, alpha, trace_grid, s, S, P, st); });
            HIP_TRY(c, kt.end());
            HIP_TRY(c, kt.begin(VVPT_K_EXTEND));
            with_stack(STACK, [&](auto k) { launch_extend<decltype(k)::value, M>(count_nodes, trace_grid, s, S, P, st, cur); });
            HIP_TRY(c, kt.end());
            HIP_TRY(c, kt.begin(VVPT_K_SHADE));
            with_features<M>(fx, [&](auto f) {
                hipLaunchKernelGGL((k_shade<M, decltype(f)>), g_shade, dim3(kBlock), 0, s, ShadeArgs{S, P, st, cur});
            });
            HIP_TRY(c, kt.end());
            if (P.nrc_use) {
                /* cache queries of this iteration: gather, infer, add throughput x radiance */
                HIP_TRY(c, kt.begin(VVPT_K_NRC));
                hipLaunchKernelGGL(k_nrc_gather, g_shade, dim3(kBlock), 0, s, P, st);
                const std::string e = c->nrc->infer_dev(P.nrc_qin, P.nrc_ctr + 2, nslots, P.nrc_qpred, cus * kNrcInferBlocksPerCU,
                                                                 cus * kNrcEncodeBlocksPerCU);
                if (!e.empty()) return set_err(c, VVPT_DEVICE_LOST, "NRC inference: " + e);
                hipLaunchKernelGGL(k_nrc_apply, g_shade, dim3(kBlock), 0, s, P, st);
                HIP_TRY(c, kt.end());
            }
            return VVPT_OK;
        };
        /* four iterations (the extension queues swap every iteration, so four leave them as they were), eager or
         * replayed from a HIP graph captured once per window */
        auto group = [&](auto mt) -> vvpt_status {
            for (uint32_t k = 0; k < 4; ++k) {
                const vvpt_status v = iteration(mt, k & 1u);
                if (v != VVPT_OK) return v;
            }
            return VVPT_OK;
        };
        const uint64_t max_iters = window_bound(nb);
        auto run_window = [&](auto mt) -> vvpt_status {
            constexpr bool M = decltype(mt)::value;
            uint64_t window_iters = 0;
            with_features<M>(fx, [&](auto f) {
                using Fi = Features<decltype(f)::ext, decltype(f)::nrc, false, true>;
                hipLaunchKernelGGL((k_init<M, Fi>), dim3((P.nslots + kBlock - 1) / kBlock), dim3(kBlock), 0, s, S, P, st);
            });
            hipGraphExec_t gx = nullptr;
            if (graph) {
                hipGraph_t g = nullptr;
                HIP_TRY(c, hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal));
                const vvpt_status v = group(mt);
                const hipError_t e = hipStreamEndCapture(s, &g);
                if (v != VVPT_OK) {
                    if (g) (void)hipGraphDestroy(g);
                    return v;
                }
                HIP_TRY(c, e);
                const hipError_t ei = hipGraphInstantiate(&gx, g, nullptr, nullptr, 0);
                (void)hipGraphDestroy(g);
                HIP_TRY(c, ei);
            }
            vvpt_status v = VVPT_OK;
            for (;;) {
                if (gx) {
                    const hipError_t e = hipGraphLaunch(gx, s);
                    if (e != hipSuccess) {
                        v = set_err(c, VVPT_DEVICE_LOST, std::string("hipGraphLaunch: ") + hipGetErrorString(e));
                        break;
                    }
                } else {
                    v = group(mt);
                    if (v != VVPT_OK) break;
                }
                iterations += 4;
                window_iters += 4;
                hipError_t e = hipMemcpyAsync(c->h_counters, cb, kCounterBytes, hipMemcpyDeviceToHost, s);
                if (e == hipSuccess) e = hipStreamSynchronize(s);
                if (e != hipSuccess) {
                    v = set_err(c, VVPT_DEVICE_LOST, std::string("counter readback: ") + hipGetErrorString(e));
                    break;
                }
                uint64_t active = 0, started = 0;
                const uint32_t *extc = c->h_counters + (size_t)CB_EXT0 * kShards * kPad;
                const uint32_t *itc = c->h_counters + (size_t)CB_ITEMS * kShards * kPad;
                for (uint32_t sh = 0; sh < kShards; ++sh) {
                    active += extc[sh * kPad];
                    const uint32_t skip = P.items_per_shard - item_shard_size(P.items_total, P.items_per_shard, P.item_chunk, sh);
                    started += std::min<uint32_t>(itc[sh * kPad], P.items_per_shard) - skip;
                }
                const uint64_t done = items_done_before + (started > active ? started - active : 0);
                c->progress.store((float)((double)done / (double)total_items));
                if (active == 0u) break;
                if (!gx) { /* a captured graph keeps its grids */
                    live = (uint32_t)std::min<uint64_t>(active, P.nslots);
                    size_grids();
                }
                if (window_iters >= max_iters) {
                    v = set_err(c, VVPT_TIMEOUT, "render did not finish within " + std::to_string(max_iters) +
                                                     " wavefront iterations");
                    break;
                }
            }
            if (gx) (void)hipGraphExecDestroy(gx);
            return v;
        };
        const vvpt_status vw = multi ? run_window(std::true_type()) : run_window(std::false_type());
        if (vw != VVPT_OK) return vw;
        if (!multi) {
            hipLaunchKernelGGL(k_resolve, dim3((J[0].npix + kBlock - 1) / kBlock), dim3(kBlock), 0, s, P, S.job, nb,
                               w == 0 ? 1u : 0u, (float4 *)jobs[0].rad, (float4 *)jobs[0].alb, (float4 *)jobs[0].nrm);
            items_done_before += (uint64_t)nb * J[0].npix;
        } else {
            for (size_t i = 0; i < njobs; ++i)
                if (dindex[i] >= 0)
                    hipLaunchKernelGGL(k_resolve, dim3((J[i].npix + kBlock - 1) / kBlock), dim3(kBlock), 0, s, P, J[i],
                                       batches[i], 1u, (float4 *)jobs[i].rad, (float4 *)nullptr, (float4 *)nullptr);
            items_done_before += total_items;
        }
        if (nrc && w + 1 < wins.size()) {
            /* train on this frame's samples: Adam steps over batches of 16384.  Not after the last frame: every
             * render starts from the cache's initial state, so that training could not change any output */
            uint32_t hc[2];
            HIP_TRY(c, hipMemcpyAsync(hc, P.nrc_ctr, sizeof(hc), hipMemcpyDeviceToHost, s));
            HIP_TRY(c, hipStreamSynchronize(s));
            const uint32_t nt = (flags & VVPT_FLAG_NRC_UNTRAINED) ? 0u : std::min(hc[1], P.nrc_tcap);
            const uint32_t epochs = opt.nrc_epochs ? opt.nrc_epochs : 1u;
            const uint32_t nrc_step = opt.nrc_step_samples
                                          ? std::min(NrcModel::kMaxBatch, std::max(1024u, opt.nrc_step_samples / 64u * 64u))
                                          : 16384u;
            HIP_TRY(c, kt.begin(VVPT_K_NRC));
            for (uint32_t ep = 0; ep < epochs; ++ep)
            for (uint32_t o = 0; o + 1024 <= nt; o += nrc_step) {
                const uint32_t m = std::min(nrc_step, nt - o);
                /* with the fallback on, every 8th sample of the frame is held out of training to judge the cache */
                const std::string e = c->nrc->train_step(P.nrc_tin + (size_t)o * 10, P.nrc_ttgt + (size_t)o * 3, m,
                                                         nullptr, P.nrc_ok ? (int64_t)o : -1);
                if (!e.empty()) return set_err(c, VVPT_DEVICE_LOST, "NRC training: " + e);
                nrc_trained += m;
            }
            if (P.nrc_ok && nt > 0) {
                std::string e = c->nrc->evaluate_holdout(P.nrc_tin, P.nrc_ttgt, nt);
                if (!e.empty()) return set_err(c, VVPT_DEVICE_LOST, "NRC error estimate: " + e);
                /* a cell serves queries with at least 16 samples behind it and an error sum within the tolerance of
                 * the target sum plus two standard deviations of the targets' noise; older frames count half */
                e = c->nrc->error_flags(opt.nrc_tolerance > 0.0f ? opt.nrc_tolerance : 0.05f, 2.0f, 16.0f, 0.5f);
                if (!e.empty()) return set_err(c, VVPT_DEVICE_LOST, "NRC error estimate: " + e);
            }
            HIP_TRY(c, kt.end());
        }
    }
    HIP_TRY(c, hipEventRecord(c->ev1, s));
    HIP_TRY(c, hipGetLastError());
    HIP_TRY(c, hipStreamSynchronize(s));
    c->progress.store(1.0f);
    if (multi && done_ms) {
        /* completion times: device wall-clock ticks since the start stamp */
        const size_t nj = djobs.size();
        std::vector<unsigned long long> ticks(nj + 1);
        HIP_TRY(c, hipMemcpy(ticks.data(), d_ticks, (nj + 1) * 8, hipMemcpyDeviceToHost));
        int khz = 0;
        HIP_TRY(c, hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, c->device));
        for (size_t i = 0; i < njobs; ++i)
            if (dindex[i] >= 0 && khz > 0) {
                const unsigned long long t = ticks[(size_t)dindex[i]], t0 = ticks[nj];
                done_ms[i] = t >= t0 ? (double)(t - t0) / (double)khz : 0.0;
            }
    }
    if (stats) {
        std::vector<unsigned long long> hsh((size_t)kShards * kStatStride);
        HIP_TRY(c, hipMemcpy(hsh.data(), c->stats.p, hsh.size() * sizeof(unsigned long long), hipMemcpyDeviceToHost));
        unsigned long long hs[S_NSTATS] = {0};
        for (uint32_t sh = 0; sh < kShards; ++sh)
            for (uint32_t k = 0; k < S_NSTATS; ++k) hs[k] += hsh[(size_t)sh * kStatStride + k];
        float ms = 0.0f;
        HIP_TRY(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
        std::memset(stats, 0, sizeof(*stats));
        stats->path_rays = hs[S_PATH];
        stats->shadow_rays = hs[S_SHADOW] + hs[S_SHADOW_SEC];
        stats->nee_rays = hs[S_NEE];
        stats->iterations = iterations;
        stats->render_ms = ms;
        stats->nodes[VVPT_K_EXTEND] = hs[S_NODES_EXT];
        stats->tris[VVPT_K_EXTEND] = hs[S_TRIS_EXT];
        stats->nodes[VVPT_K_SECONDARY] = hs[S_NODES_SEC];
        stats->tris[VVPT_K_SECONDARY] = hs[S_TRIS_SEC];
        stats->nodes[VVPT_K_SHADOW] = hs[S_NODES_SHD];
        stats->tris[VVPT_K_SHADOW] = hs[S_TRIS_SHD];
        stats->nrc_queries = hs[S_NRCQ];
        stats->nrc_fallbacks = hs[S_NRC_FALLBACK];
        stats->nrc_train_samples = nrc_trained;
        if (nrc && nrc_trained) {
            float lo = 0.0f;
            HIP_TRY(c, hipMemcpy(&lo, c->nrc->loss, sizeof(float), hipMemcpyDeviceToHost));
            stats->nrc_loss = lo;
        }
        HIP_TRY(c, kt.collect(stats));
    }
    return VVPT_OK;
}

vvpt_status check_info(vvpt_ctx *c, const vvpt_render_info *info) {
    if (!info || info->width == 0 || info->height == 0 || info->batch_size == 0 || info->depth == 0)
        return set_err(c, VVPT_INVALID, "invalid render info");
    if (info->batch_size > 0xffffu || info->depth > 255u) return set_err(c, VVPT_INVALID, "batch size or depth too large");
    if ((uint64_t)info->width * info->height > (1ull << 28)) return set_err(c, VVPT_INVALID, "resolution too large");
    return VVPT_OK;
}

}  // namespace

extern "C" {

}  // extern "C"

namespace {

/* Bodies of the render and denoise entry points; the caller has taken the context. */
vvpt_status render_device_taken(vvpt_ctx *c, const vvpt_render_info *info, float *d_rad, float *d_alb, float *d_nrm,
                                void *stream, vvpt_stats *stats) {
    vvpt_status v = check_info(c, info);
    if (v != VVPT_OK) return v;
    if (!d_rad) return set_err(c, VVPT_INVALID, "null radiance buffer");
    if ((info->flags & VVPT_FLAG_AOVS) && (!d_alb || !d_nrm)) return set_err(c, VVPT_INVALID, "null AOV buffer");
    if (!c->sh.valid || c->sh.num_instances == 0) return set_err(c, VVPT_WARN_EMPTY_SCENE, "Trying to render an empty scene");
    HIP_TRY(c, hipSetDevice(c->device));
    hipStream_t s = stream ? (hipStream_t)stream : c->stream;
    const std::vector<JobSpec> jobs = {{0u, *info, d_rad, d_alb, d_nrm}};
    return render_core(c, jobs, false, info->flags, s, stats, nullptr);
}

vvpt_status render_jobs_taken(vvpt_ctx *c, vvpt_job *jobs, uint32_t count, uint32_t flags, void *stream,
                              vvpt_stats *stats) {
    if (!jobs || count == 0 || count > VVPT_MAX_JOBS) return set_err(c, VVPT_INVALID, "job count out of range");
    if (flags & (VVPT_FLAG_AOVS | VVPT_FLAG_NRC))
        return set_err(c, VVPT_UNSUPPORTED, "AOVs and the radiance cache are single-render features");
    if (!c->sh.valid || c->sh.num_instances == 0) return set_err(c, VVPT_WARN_EMPTY_SCENE, "Trying to render an empty scene");
    std::vector<JobSpec> js(count);
    for (uint32_t i = 0; i < count; ++i) {
        vvpt_status v = check_info(c, &jobs[i].info);
        if (v != VVPT_OK) return v;
        if (!jobs[i].d_radiance_rgba) return set_err(c, VVPT_INVALID, "null radiance buffer");
        if (jobs[i].scene >= c->sh.parts.size()) return set_err(c, VVPT_INVALID, "job references a missing scene");
        js[i] = {jobs[i].scene, jobs[i].info, jobs[i].d_radiance_rgba, nullptr, nullptr};
        jobs[i].done_ms = 0.0;
    }
    HIP_TRY(c, hipSetDevice(c->device));
    hipStream_t s = stream ? (hipStream_t)stream : c->stream;
    std::vector<double> done(count, 0.0);
    const vvpt_status v = render_core(c, js, true, flags, s, stats, done.data());
    if (v != VVPT_OK) return v;
    for (uint32_t i = 0; i < count; ++i) jobs[i].done_ms = done[i];
    return VVPT_OK;
}

vvpt_status denoise_device_taken(vvpt_ctx *c, const float *d_rad, const float *d_alb, const float *d_nrm, uint32_t W,
                                 uint32_t H, float *d_out, void *stream) {
    if (!d_rad || !d_alb || !d_nrm || !d_out || W == 0 || H == 0 || (uint64_t)W * H > (1ull << 28))
        return set_err(c, VVPT_INVALID, "denoise: invalid image");
    HIP_TRY(c, hipSetDevice(c->device));
    hipStream_t s = stream ? (hipStream_t)stream : c->stream;
    HIP_TRY(c, ensure(c->dnbuf, (size_t)W * H * 32));
    const std::string e = denoise_device(d_rad, d_alb, d_nrm, W, H, d_out, (float *)c->dnbuf.p, s);
    if (!e.empty()) return set_err(c, VVPT_DEVICE_LOST, "denoise: " + e);
    HIP_TRY(c, hipStreamSynchronize(s));
    return VVPT_OK;
}

}  // namespace

extern "C" {

vvpt_status vvpt_render_device(vvpt_ctx *c, const vvpt_render_info *info, float *d_rad, float *d_alb, float *d_nrm,
                               void *stream, vvpt_stats *stats) {
    if (!c) return VVPT_INVALID;
    VVPT_TAKE(c);
    return render_device_taken(c, info, d_rad, d_alb, d_nrm, stream, stats);
}

vvpt_status vvpt_render_jobs(vvpt_ctx *c, vvpt_job *jobs, uint32_t count, uint32_t flags, void *stream,
                             vvpt_stats *stats) {
    if (!c) return VVPT_INVALID;
    VVPT_TAKE(c);
    return render_jobs_taken(c, jobs, count, flags, stream, stats);
}

vvpt_status vvpt_denoise_device(vvpt_ctx *c, const float *d_rad, const float *d_alb, const float *d_nrm, uint32_t W,
                                uint32_t H, float *d_out, void *stream) {
    if (!c) return VVPT_INVALID;
    VVPT_TAKE(c);
    return denoise_device_taken(c, d_rad, d_alb, d_nrm, W, H, d_out, stream);
}

vvpt_status vvpt_denoise_device_noalloc(vvpt_ctx *c, const float *d_rad, const float *d_alb, const float *d_nrm,
                                        uint32_t W, uint32_t H, float *d_out, void *stream) {
    if (!c) return VVPT_INVALID;
    VVPT_TAKE(c);
    if (!d_rad || !d_alb || !d_nrm || !d_out || W == 0 || H == 0)
        return set_err(c, VVPT_INVALID, "denoise: invalid image");
    if ((uint64_t)W * H > kDenoiseScratchPixels)
        return set_err(c, VVPT_INVALID, "denoise: " + std::to_string((uint64_t)W * H) + " pixels exceed the " +
                                            std::to_string(kDenoiseScratchPixels) +
                                            "-pixel limit of the allocation-free denoise");
    HIP_TRY(c, hipSetDevice(c->device));
    hipStream_t s = stream ? (hipStream_t)stream : c->stream;
    const std::string e = denoise_device_noalloc(d_rad, d_alb, d_nrm, W, H, d_out, c->device, s);
    if (!e.empty()) return set_err(c, VVPT_DEVICE_LOST, "denoise: " + e);
    return VVPT_OK;
}

vvpt_status vvpt_denoise(vvpt_ctx *c, const float *rad, const float *alb, const float *nrm, uint32_t W, uint32_t H,
                         float *out) {
    if (!c) return VVPT_INVALID;
    VVPT_TAKE(c);
    if (!rad || !alb || !nrm || !out || W == 0 || H == 0 || (uint64_t)W * H > (1ull << 28))
        return set_err(c, VVPT_INVALID, "denoise: invalid image");
    HIP_TRY(c, hipSetDevice(c->device));
    const size_t bytes = (size_t)W * H * 16;
    HIP_TRY(c, ensure(c->dnio, 3 * bytes));
    float *d = (float *)c->dnio.p;
    HIP_TRY(c, hipMemcpy(d, rad, bytes, hipMemcpyHostToDevice));
    HIP_TRY(c, hipMemcpy(d + (size_t)W * H * 4, alb, bytes, hipMemcpyHostToDevice));
    HIP_TRY(c, hipMemcpy(d + (size_t)W * H * 8, nrm, bytes, hipMemcpyHostToDevice));
    const vvpt_status v = denoise_device_taken(c, d, d + (size_t)W * H * 4, d + (size_t)W * H * 8, W, H, d, nullptr);
    if (v != VVPT_OK) return v;
    HIP_TRY(c, hipMemcpy(out, d, bytes, hipMemcpyDeviceToHost));
    return VVPT_OK;
}

vvpt_status vvpt_set_tuning(vvpt_ctx *c, const vvpt_tuning *t) {
    if (!c || !t) return VVPT_INVALID;
    VVPT_TAKE(c);
    if (t->slots < 64u || t->slots > (1u << 27) || t->trace_blocks_per_cu < 1u || t->trace_blocks_per_cu > 64u ||
        t->shade_blocks_per_cu < 1u || t->shade_blocks_per_cu > 1024u)
        return set_err(c, VVPT_INVALID, "tuning out of range");
    c->tune = *t;
    return VVPT_OK;
}

vvpt_status vvpt_get_tuning(const vvpt_ctx *c, vvpt_tuning *t) {
    if (!c || !t) return VVPT_INVALID;
    *t = c->tune;
    return VVPT_OK;
}

vvpt_status vvpt_set_options(vvpt_ctx *c, const vvpt_options *o) {
    if (!c || !o) return VVPT_INVALID;
    VVPT_TAKE(c);
    if (!std::isfinite(o->nrc_spread) || o->nrc_spread < 0.0f || !std::isfinite(o->nrc_tolerance) ||
        o->nrc_frame_batches > 0xffffu || o->nrc_epochs > 64u)
        return set_err(c, VVPT_INVALID, "options out of range");
    c->opt = *o;
    return VVPT_OK;
}

vvpt_status vvpt_get_options(const vvpt_ctx *c, vvpt_options *o) {
    if (!c || !o) return VVPT_INVALID;
    *o = c->opt;
    return VVPT_OK;
}

vvpt_status vvpt_autotune(vvpt_ctx *c, vvpt_job *probe, uint32_t count, uint32_t flags, vvpt_tuning *best,
                          double *best_ms) {
    if (!c || !probe || count == 0) return c ? set_err(c, VVPT_INVALID, "empty probe") : VVPT_INVALID;
    VVPT_TAKE(c);
    flags &= ~(uint32_t)(VVPT_FLAG_KERNEL_TIMING | VVPT_FLAG_COUNT_NODES);
    int reps = 2;
    auto time_of = [&](const vvpt_tuning &t, double &ms) -> vvpt_status {
        c->tune = t;
        ms = 1e300;
        for (int r = 0; r < reps; ++r) {
            vvpt_stats st;
            const vvpt_status e = render_jobs_taken(c, probe, count, flags, nullptr, &st);
            if (e != VVPT_OK) return e;
            ms = std::min(ms, st.render_ms);
        }
        return VVPT_OK;
    };
    const vvpt_tuning start = c->tune;
    vvpt_tuning cur = start;
    double cur_ms = 0.0;
    vvpt_status v = time_of(cur, cur_ms); /* also the warm-up (buffers grow on first use) */
    if (v != VVPT_OK) return v;
    if (cur_ms >= 100.0) reps = 1;
    if ((v = time_of(cur, cur_ms)) != VVPT_OK) return v;
    auto sweep = [&](uint32_t vvpt_tuning::*field, std::initializer_list<uint32_t> values) -> vvpt_status {
        for (uint32_t x : values) {
            if (cur.*field == x) continue;
            vvpt_tuning t = cur;
            t.*field = x;
            double ms = 0.0;
            const vvpt_status e = time_of(t, ms);
            if (e != VVPT_OK) {
                c->tune = cur;
                return e;
            }
            if (ms < cur_ms) {
                cur = t;
                cur_ms = ms;
            }
        }
        return VVPT_OK;
    };
    if ((v = sweep(&vvpt_tuning::slots, {1u << 21, 1u << 22, 1u << 23, 1u << 24, 1u << 25})) != VVPT_OK) return v;
    if ((v = sweep(&vvpt_tuning::trace_blocks_per_cu, {8u, 12u, 16u, 24u, 32u})) != VVPT_OK) return v;
    if ((v = sweep(&vvpt_tuning::shade_blocks_per_cu, {16u, 32u, 64u, 128u})) != VVPT_OK) return v;
    c->tune = cur;
    if (best) *best = cur;
    if (best_ms) *best_ms = cur_ms;
    return VVPT_OK;
}

vvpt_status vvpt_render(vvpt_ctx *c, const vvpt_render_info *info, float *rad, float *alb, float *nrm, vvpt_stats *stats) {
    if (!c) return VVPT_INVALID;
    VVPT_TAKE(c);
    vvpt_status v = check_info(c, info);
    if (v != VVPT_OK) return v;
    if (!rad) return set_err(c, VVPT_INVALID, "null radiance buffer");
    HIP_TRY(c, hipSetDevice(c->device));
    const size_t npix = (size_t)info->width * info->height;
    const bool want_aovs = alb != nullptr || nrm != nullptr;
    vvpt_render_info ri = *info;
    if (want_aovs) ri.flags |= VVPT_FLAG_AOVS;
    HIP_TRY(c, ensure(c->outputs, npix * 16 * 3));
    float *d = (float *)c->outputs.p;
    v = render_device_taken(c, &ri, d, d + npix * 4, d + npix * 8, nullptr, stats);
    if (v != VVPT_OK) return v;
    HIP_TRY(c, hipMemcpy(rad, d, npix * 16, hipMemcpyDeviceToHost));
    if (alb) HIP_TRY(c, hipMemcpy(alb, d + npix * 4, npix * 16, hipMemcpyDeviceToHost));
    if (nrm) HIP_TRY(c, hipMemcpy(nrm, d + npix * 8, npix * 16, hipMemcpyDeviceToHost));
    return VVPT_OK;
}

vvpt_status vvpt_trace_primary(vvpt_ctx *c, const vvpt_render_info *info, uint32_t *inst, uint32_t *prim, float *t,
                               float *u, float *v) {
    if (!c || !info || !inst || !prim || !t || !u || !v) return VVPT_INVALID;
    VVPT_TAKE(c);
    vvpt_status vs = check_info(c, info);
    if (vs != VVPT_OK) return vs;
    if (!c->sh.valid || c->sh.num_instances == 0) return set_err(c, VVPT_WARN_EMPTY_SCENE, "empty scene");
    HIP_TRY(c, hipSetDevice(c->device));
    DScene S;
    vs = make_dscene(c, false, S);
    if (vs == VVPT_OK) vs = make_jobview(c, 0u, *info, false, S.job);
    if (vs != VVPT_OK) return vs;
    const uint32_t n = info->width * info->height;
    DevBuf out;
    HIP_TRY(c, ensure(out, (size_t)n * 20));
    uint32_t *di = (uint32_t *)out.p, *dp = di + n;
    float *dt = (float *)(dp + n), *du = dt + n, *dv = du + n;
    const int STACK = stack_size_for(c->sh.max_depth);
    dim3 grid((n + kTraceBlock - 1) / kTraceBlock);
    hipStream_t s = c->stream;
    if (!with_stack(STACK, [&](auto k) {
            hipLaunchKernelGGL((k_trace_primary<decltype(k)::value>), grid, dim3(kTraceBlock), 0, s, S, info->width,
                               info->height, info->seed, di, dp, dt, du, dv);
        })) {
        release(out);
        return set_err(c, VVPT_UNSUPPORTED, "BVH too deep");
    }
    hipError_t e = hipStreamSynchronize(s);
    if (e == hipSuccess) e = hipMemcpy(inst, di, n * 4, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(prim, dp, n * 4, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(t, dt, n * 4, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(u, du, n * 4, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(v, dv, n * 4, hipMemcpyDeviceToHost);
    release(out);
    if (e != hipSuccess) return set_err(c, VVPT_DEVICE_LOST, hipGetErrorString(e));
    return VVPT_OK;
}

}  // extern "C"
