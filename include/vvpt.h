/*
 * vvpt.h - C ABI of the MI355X (gfx950) path tracer.
 *
 * This is the drop-in boundary for the path-tracing renderer of vengine
 * (kwstanths/vviewer).  The reference boundary is the C++ abstract class
 * vengine::RendererPathTracing (src/lib/vengine/core/Renderer.hpp:11-39):
 *     RenderInfo { samples, depth, batchSize, filename, fileType, exposure,
 *                  width, height, denoise, writeAllFiles }     (:14-28)
 *     bool  isRayTracingEnabled();                             (:33)
 *     void  render();                                          (:34)
 *     float renderProgress();                                  (:35)
 * whose inputs are read implicitly from the engine's Scene (camera, environment,
 * objects with mesh/material/light/volume components).  Here those inputs are
 * explicit: the caller describes the scene once with vvpt_set_scene() and then
 * calls vvpt_render() with the RenderInfo fields.  The output is the
 * accumulated FP32 RGBA radiance buffer that the reference reads back in
 * VulkanRendererPathTracing::getRenderTargetData (VulkanRendererPathTracing.cpp:903-956):
 * row-major, top row first, A = 1, already divided by the total sample count.
 *
 * Conventions: plain C99 types only; no exceptions cross this boundary; every
 * call returns a vvpt_status; one render in flight per context (VVPT_BUSY
 * otherwise).  The library copies all scene data in vvpt_set_scene(); the
 * caller may free its arrays after the call returns.
 */
#ifndef VVPT_H
#define VVPT_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define VVPT_ABI_VERSION 4u

typedef struct vvpt_ctx vvpt_ctx;

typedef enum {
    VVPT_OK = 0,
    VVPT_WARN_EMPTY_SCENE = 1, /* reference: ConsoleWarning + return (VulkanRendererPathTracing.cpp:133-136) */
    VVPT_TIMEOUT = -1,         /* reference: VK_TIMEOUT on the per-batch fence (:869-876) */
    VVPT_DEVICE_LOST = -2,     /* reference: VK_ERROR_DEVICE_LOST (:877-882) */
    VVPT_INVALID = -3,
    VVPT_OOM = -4,
    VVPT_BUSY = -5,            /* reference: m_renderInProgress guard (:123-124) */
    VVPT_UNSUPPORTED = -6,     /* reference: isRayTracingEnabled() == false (VulkanRenderer.cpp:106-111) */
    VVPT_NOT_BUILT = -7        /* the HIP code object for gfx950 is missing */
} vvpt_status;

/* ---------------------------------------------------------------- scene -- */

/* Vertex: mirrors vengine::Vertex (core/Mesh.hpp:15-21, shaders/include/structs.glsl:4-12), 68 bytes. */
typedef struct {
    float position[3];
    float uv[2];
    float normal[3];
    float color[3];
    float tangent[3];
    float bitangent[3];
} vvpt_vertex;

typedef struct {
    const vvpt_vertex *vertices;
    uint32_t num_vertices;
    const uint32_t *indices; /* 3 * num_triangles vertex indices (reference: u32 index buffer, VulkanMesh.cpp:15-26) */
    uint32_t num_triangles;
} vvpt_mesh;

/* One scene object with a mesh.  Mirrors InstanceData (core/Instances.hpp:17-35):
 * model matrix, material index, front/back facing volume material (-1 = none). */
typedef struct {
    float transform[12];  /* object-to-world, row-major 3x4 (rows of the model matrix) */
    uint32_t mesh;
    uint32_t material;
    int32_t front_volume; /* InstanceData.id.g */
    int32_t back_volume;  /* InstanceData.id.b */
} vvpt_instance;

typedef enum {
    VVPT_MATERIAL_PBR_STANDARD = 0, /* MaterialType::MATERIAL_PBR_STANDARD */
    VVPT_MATERIAL_LAMBERT = 1,      /* MaterialType::MATERIAL_LAMBERT */
    VVPT_MATERIAL_VOLUME = 2        /* MaterialType::MATERIAL_VOLUME */
} vvpt_material_type;

#define VVPT_TEXTURE_DEFAULT (-1)

/* Mirrors MaterialData (shaders/include/structs.glsl:41-52) before texture
 * binding.  Volume materials reuse the block like VulkanMaterialVolume
 * (VulkanMaterial.cpp:449-481): sigma_a = albedo.rgb, sigma_s = (metallic,
 * roughness, ao), g = emissive[0]. Texture ids index vvpt_scene_desc.textures;
 * VVPT_TEXTURE_DEFAULT selects the reference's default texture for that slot
 * (white / whiteColor / normalmapdefault, VulkanMaterial.cpp:30-62,222-250). */
typedef struct {
    uint32_t type;        /* vvpt_material_type */
    float albedo[4];      /* rgb, alpha */
    float metallic, roughness, ao;
    float transparent;    /* 0 or 1 (metallicRoughnessAO.a, VulkanMaterial.cpp:76) */
    float emissive[4];    /* rgb, intensity */
    int32_t tex_albedo, tex_metallic, tex_roughness, tex_ao, tex_emissive, tex_normal, tex_alpha;
    float uv_tiling[2];
} vvpt_material;

typedef enum {
    VVPT_TEXTURE_RGBA8_UNORM = 0,
    VVPT_TEXTURE_RGBA8_SRGB = 1,
    VVPT_TEXTURE_RGBA32F = 2
} vvpt_texture_format;

typedef struct {
    uint32_t width, height;
    uint32_t format;   /* vvpt_texture_format */
    const void *data;  /* width*height texels, row 0 first */
} vvpt_texture;

typedef enum {
    VVPT_LIGHT_POINT = 0,       /* LightType::POINT_LIGHT */
    VVPT_LIGHT_DIRECTIONAL = 1  /* LightType::DIRECTIONAL_LIGHT */
} vvpt_light_type;

/* Mirrors LightData + LightInstance (structs.glsl:55-69, VulkanInstances.cpp:71-90).
 * point: position = world position.  directional: position = world +Z axis of
 * the light object (modelMatrix * (0,0,1,0)); light arrives from -position.
 * Mesh lights are not listed here: every instance whose material is emissive
 * becomes one (core/Instances.cpp:112-114, Material.cpp:85-88). */
typedef struct {
    uint32_t type;
    float color[4]; /* rgb, intensity */
    float position[3];
} vvpt_light;

typedef enum { VVPT_CAMERA_PERSPECTIVE = 0, VVPT_CAMERA_ORTHOGRAPHIC = 1 } vvpt_camera_type;

/* Mirrors Camera (core/Camera.hpp:20-105) as used by render() (VulkanRendererPathTracing.cpp:143-194). */
typedef struct {
    uint32_t type;
    float view[16];       /* world-to-camera, column-major (glm layout) */
    float fov_degrees;    /* vertical field of view (perspective) */
    float ortho_width, ortho_height;
    float znear, zfar;
    float lens_radius, focal_distance;
    int32_t volume;       /* material index of the camera's volume or -1 */
} vvpt_camera;

typedef enum {
    VVPT_ENV_SOLID_COLOR = 0,
    VVPT_ENV_HDRI = 1,
    VVPT_ENV_SOLID_COLOR_WITH_HDRI_LIGHTING = 2
} vvpt_environment_type;

typedef struct {
    uint32_t type;            /* vvpt_environment_type (Scene.hpp:19-24) */
    float background[3];
    float intensity;          /* environment map intensity */
    int32_t equirect_texture; /* RGBA32F equirectangular map or -1 */
} vvpt_environment;

typedef struct {
    const vvpt_mesh *meshes;         uint32_t num_meshes;
    const vvpt_instance *instances;  uint32_t num_instances;
    const vvpt_material *materials;  uint32_t num_materials;
    const vvpt_texture *textures;    uint32_t num_textures;
    const vvpt_light *lights;        uint32_t num_lights;
    vvpt_camera camera;
    vvpt_environment environment;
} vvpt_scene_desc;

/* ---------------------------------------------------------------- render -- */

typedef enum {
    VVPT_FLAG_AOVS = 1u << 0,          /* also accumulate first-hit albedo and normal (outputImage[1..2]) */
    VVPT_FLAG_EXTENDED = 1u << 1,      /* extended estimator, not the reference's stream: scrambled Sobol samples
                                          and, with an HDRI environment, importance sampling of the environment
                                          with multiple importance sampling; converges to the same image */
    VVPT_FLAG_KERNEL_TIMING = 1u << 2, /* time every kernel launch with hipEvents (vvpt_stats.kernel_ms) */
    VVPT_FLAG_COUNT_NODES = 1u << 3,   /* count node visits and triangle tests (vvpt_stats.nodes/.tris) */
    VVPT_FLAG_NRC = 1u << 4,           /* extended estimator with the neural radiance cache: frames of 4 batches;
                                          a hashed fraction of samples trains the cache (online, after each frame
                                          but the last; the cache starts from its initial state in every render),
                                          the other paths end in a cache query once their spread exceeds the
                                          primary footprint (from the second frame on) */
    VVPT_FLAG_GRAPH = 1u << 5,         /* replay the wavefront loop from a HIP graph of four iterations, captured
                                          once per launch window (not with VVPT_FLAG_NRC or _KERNEL_TIMING);
                                          the result is identical to the eager loop's */
    VVPT_FLAG_NRC_UNTRAINED = 1u << 6  /* with VVPT_FLAG_NRC: the cache keeps its initial state (no training steps
                                          after frames), the control against which training is measured */
} vvpt_render_flags;

/* RenderInfo fields that reach the device path (core/Renderer.hpp:14-28). */
typedef struct {
    uint32_t samples;     /* total samples per pixel; samples % batch_size is dropped like the reference (:798-799) */
    uint32_t depth;       /* max path depth */
    uint32_t batch_size;  /* samples per batch; the RNG restarts per batch */
    uint32_t width, height;
    uint32_t seed;        /* 0 = the reference stream */
    uint32_t flags;       /* vvpt_render_flags */
} vvpt_render_info;

/* Per-render counters, filled by vvpt_render*(). */
typedef enum {
    VVPT_K_EXTEND = 0,    /* closest-hit extension of path rays */
    VVPT_K_SHADE = 1,     /* one bounce of the hit / miss shaders; sample ends, work-item refill, queue compaction */
    VVPT_K_SECONDARY = 2, /* emitter lookups and multi-segment shadow walks */
    VVPT_K_FINISH = 3,    /* no launches of its own any more (its work is in VVPT_K_SHADE): always 0 */
    VVPT_K_SHADOW = 4,    /* single-segment shadow rays */
    VVPT_K_NRC = 5,       /* radiance-cache queries and training */
    VVPT_K_COUNT = 6
} vvpt_kernel;

typedef struct {
    uint64_t path_rays;       /* closest-hit extension rays */
    uint64_t shadow_rays;     /* light-sampling visibility segments */
    uint64_t nee_rays;        /* BSDF-direction emitter lookups that needed their own traversal */
    uint64_t iterations;      /* wavefront iterations */
    double   render_ms;       /* device time of the render loop (hipEvents) */
    double   kernel_ms[VVPT_K_COUNT];        /* VVPT_FLAG_KERNEL_TIMING: summed launch durations */
    uint64_t kernel_launches[VVPT_K_COUNT];
    uint64_t nodes[VVPT_K_COUNT];             /* VVPT_FLAG_COUNT_NODES: wide-node visits per kernel */
    uint64_t tris[VVPT_K_COUNT];              /* VVPT_FLAG_COUNT_NODES: triangle tests per kernel */
    uint64_t nrc_queries;                     /* VVPT_FLAG_NRC: paths that ended in a cache query */
    uint64_t nrc_train_samples;               /* VVPT_FLAG_NRC: training samples used */
    double   nrc_loss;                        /* VVPT_FLAG_NRC: loss of the last training step */
    uint64_t nrc_fallbacks;                   /* VVPT_FLAG_NRC: paths that would have ended in a query but went on,
                                                 because the cache's error estimate there exceeds its tolerance */
} vvpt_stats;

uint32_t    vvpt_abi_version(void);
vvpt_status vvpt_create(vvpt_ctx **out, int hip_device);
void        vvpt_destroy(vvpt_ctx *ctx);
/* reference: isRayTracingEnabled() (Renderer.hpp:33) */
int         vvpt_is_enabled(const vvpt_ctx *ctx);
vvpt_status vvpt_set_scene(vvpt_ctx *ctx, const vvpt_scene_desc *scene);
/* reference: render() (Renderer.hpp:34; VulkanRendererPathTracing.cpp:121-226,791-956).
 * Host buffers of width*height*4 floats; albedo/normal may be NULL. */
vvpt_status vvpt_render(vvpt_ctx *ctx, const vvpt_render_info *info, float *radiance_rgba,
                        float *albedo_rgba, float *normal_rgba, vvpt_stats *stats);
/* Same as vvpt_render but the outputs are device pointers on the context's
 * device (no readback); `stream` is a hipStream_t or NULL for the context's stream. */
vvpt_status vvpt_render_device(vvpt_ctx *ctx, const vvpt_render_info *info, float *d_radiance_rgba,
                               float *d_albedo_rgba, float *d_normal_rgba, void *stream, vvpt_stats *stats);
/* reference: renderProgress() (Renderer.hpp:35) - fraction of work items done; atomic. */
float       vvpt_progress(const vvpt_ctx *ctx);
const char *vvpt_last_error(const vvpt_ctx *ctx);

/* --------------------------------------------------------------- denoise -- */

/* The denoise step of a render (reference: storeToDisk with renderInfo.denoise, VulkanRendererPathTracing.cpp:
 * 985-1018, Open Image Denoise on the host with the radiance, albedo and normal images): this library's own
 * edge-avoiding a-trous wavelet filter on the GPU (Dammertz et al. 2010) over the albedo-demodulated radiance, with
 * edge-stopping weights from the normal and albedo AOVs.  Inputs are width*height RGBA float images as vvpt_render
 * returns them (the normal in its n * 0.5 + 0.5 encoding); out gets the denoised radiance, alpha 1, and may be any
 * of the three input buffers.  vvpt_denoise takes host buffers, vvpt_denoise_device device buffers on a stream (NULL:
 * the context's). */
vvpt_status vvpt_denoise(vvpt_ctx *ctx, const float *radiance_rgba, const float *albedo_rgba, const float *normal_rgba,
                         uint32_t width, uint32_t height, float *out_rgba);
vvpt_status vvpt_denoise_device(vvpt_ctx *ctx, const float *d_radiance_rgba, const float *d_albedo_rgba,
                                const float *d_normal_rgba, uint32_t width, uint32_t height, float *d_out_rgba,
                                void *stream);
/* No counterpart in the reference.  For callers that cannot allocate device memory (code under HIP graph capture,
 * serving loops, harnesses that forbid hipMalloc): vvpt_denoise_device with the same kernels and result, whose
 * scratch (two float4 images) is a fixed device array of the library instead of memory it allocates, so the call
 * allocates and frees nothing.  Limit: width * height <= 2,097,152 pixels (1920 x 1080 fits; larger images return
 * VVPT_INVALID).  The call only enqueues on `stream` (NULL: the context's) and returns without waiting; every call
 * on one GPU shares that GPU's array (64 MiB, held until the process ends), so calls that overlap on one GPU, on
 * different streams, race. */
vvpt_status vvpt_denoise_device_noalloc(vvpt_ctx *ctx, const float *d_radiance_rgba, const float *d_albedo_rgba,
                                        const float *d_normal_rgba, uint32_t width, uint32_t height, float *d_out_rgba,
                                        void *stream);

/* ---------------------------------------------------------- batched jobs -- */

/* The reference renders one scene per render() call and blocks on a fence per batch
 * (VulkanRendererPathTracing.cpp:791-901); a batch of independent render jobs runs here as one wavefront loop
 * over all their work items, so small jobs share the GPU with large ones instead of leaving it idle. */

/* Replaces the scene with `count` scenes, each keeping its own instances, lights and camera over one shared pool
 * of acceleration structures and buffers (one TLAS per scene); the environment of scenes[0] serves all of them.
 * vvpt_set_scene(ctx, s) is vvpt_set_scenes(ctx, s, 1). */
vvpt_status vvpt_set_scenes(vvpt_ctx *ctx, const vvpt_scene_desc *scenes, uint32_t count);

/* Replaces the camera of scene `scene` (0 after vvpt_set_scene, else an index of vvpt_set_scenes) and keeps
 * everything else: the reference builds its camera matrices from the scene's camera at every render
 * (VulkanRendererPathTracing.cpp:141-160), so a camera moved between renders (PtSceneBallOnPlane.cpp:40-55)
 * needs no new scene description, upload or acceleration-structure build.  camera->volume is an index into that
 * scene's own materials, as in its vvpt_scene_desc.  VVPT_INVALID for a missing scene, a bad camera type or a
 * singular view matrix. */
vvpt_status vvpt_set_camera(vvpt_ctx *ctx, uint32_t scene, const vvpt_camera *camera);

#define VVPT_MAX_JOBS 4096u
typedef struct {
    uint32_t scene;          /* index into the scenes of vvpt_set_scenes (0 after vvpt_set_scene) */
    vvpt_render_info info;   /* RenderInfo of the job; info.flags is ignored (the batch's flags apply) */
    float *d_radiance_rgba;  /* device buffer of width*height*4 floats, on the context's device */
    double done_ms;          /* out: device time from the start of the batch until the job's last sample ended */
} vvpt_job;

/* Renders every job; each job's radiance is bit-identical to vvpt_render_device of the same scene and info.
 * Jobs run cheapest first (pixels x samples x depth) and all GPU lanes serve the earliest unfinished jobs, so
 * small jobs complete early.  flags: VVPT_FLAG_EXTENDED, _KERNEL_TIMING, _COUNT_NODES, _GRAPH (AOVs and the
 * radiance cache are single-render features).  Every job's work items (pixels x batches) are in flight in one
 * launch window: at most 2^32 items, 16 bytes of partial result each (VVPT_MAX_PARTIAL_BYTES, default 32 GiB). */
vvpt_status vvpt_render_jobs(vvpt_ctx *ctx, vvpt_job *jobs, uint32_t count, uint32_t flags, void *stream,
                             vvpt_stats *stats);

/* Launch shape of the wavefront loop (no counterpart in the reference, whose driver schedules its dispatches). */
typedef struct {
    uint32_t slots;               /* path slots in flight (64 .. 2^27; default 2^25, about 15 GB) */
    uint32_t trace_blocks_per_cu; /* persistent trace kernels: blocks of 128 lanes per compute unit (1..64; 12) */
    uint32_t shade_blocks_per_cu; /* grid-stride kernels: blocks of 256 lanes per compute unit (1..1024; 64) */
} vvpt_tuning;
vvpt_status vvpt_set_tuning(vvpt_ctx *ctx, const vvpt_tuning *tuning);
vvpt_status vvpt_get_tuning(const vvpt_ctx *ctx, vvpt_tuning *tuning);

/* Render options beyond RenderInfo (no counterpart in the reference); a zero field selects the default.
 * max_iterations bounds the wavefront loop of one launch window: the reference aborts a batch whose fence does
 * not signal within 1 s (VulkanRendererPathTracing.cpp:869-876, VulkanUtils.hpp:23); here a window that has not
 * retired its work after max_iterations iterations (default: twice the longest schedule its work allows, see
 * vvpt_render_device) ends the render with VVPT_TIMEOUT.  Every launched kernel still completes; the host output
 * buffers of vvpt_render are not written, and the device outputs keep what earlier launch windows resolved (nothing
 * when the first window timed out). */
typedef struct {
    uint64_t max_partial_bytes;  /* per-batch partial results in flight (default 8 GiB; batched renders 32 GiB) */
    uint32_t max_iterations;     /* wavefront iterations per launch window before VVPT_TIMEOUT (0: derived bound) */
    uint32_t nrc_frame_batches;  /* VVPT_FLAG_NRC: batches per training frame (default 4) */
    uint32_t nrc_paths;          /* VVPT_FLAG_NRC: training paths per frame (default 0.042 per pixel in 22k..88k) */
    uint32_t nrc_train_cap;      /* VVPT_FLAG_NRC: training samples kept per frame (default 524288) */
    uint32_t nrc_step_samples;   /* VVPT_FLAG_NRC: samples per Adam step (default 16384) */
    uint32_t nrc_epochs;         /* VVPT_FLAG_NRC: passes over a frame's training samples (default 1) */
    float    nrc_spread;         /* VVPT_FLAG_NRC: a path queries the cache once spread^2 > nrc_spread x footprint
                                    (default 0.01) */
    float    nrc_tolerance;      /* VVPT_FLAG_NRC: relative error estimate above which a region falls back to the
                                    plain tracer (default 0.05; negative disables the fallback) */
    float    nrc_max_resolution; /* VVPT_FLAG_NRC: cells per axis of the finest hash-grid level (default 128) */
    float    nrc_learning_rate;  /* VVPT_FLAG_NRC: Adam learning rate (default 0.003, decaying by 0.999 per step) */
} vvpt_options;
vvpt_status vvpt_set_options(vvpt_ctx *ctx, const vvpt_options *options);
vvpt_status vvpt_get_options(const vvpt_ctx *ctx, vvpt_options *options);
/* Autotuner: renders the probe batch `probe[count]` (vvpt_render_jobs semantics and flags; a single render is a
 * batch of one job) for candidate shapes - slots 2^21..2^25, then trace blocks per CU in {8, 12, 16, 24, 32},
 * then shade blocks per CU in {16, 32, 64, 128}, one parameter at a time - and keeps the fastest (best of two renders
 * when a render takes under 100 ms).  The chosen shape is set on the context and written to `best`; best_ms
 * (may be NULL) receives its render time.  Results do not depend on the shape. */
vvpt_status vvpt_autotune(vvpt_ctx *ctx, vvpt_job *probe, uint32_t count, uint32_t flags, vvpt_tuning *best,
                          double *best_ms);

/* Primary-visibility query: one jittered camera ray per pixel for batch 0,
 * sample 0 (the same ray the first bounce traces).  Per pixel: instance index,
 * primitive index (0xffffffff on a miss), hit distance t and barycentrics u,v. */
vvpt_status vvpt_trace_primary(vvpt_ctx *ctx, const vvpt_render_info *info, uint32_t *instance,
                               uint32_t *primitive, float *t, float *u, float *v);

/* Acceleration-structure statistics of the current scene. */
typedef struct {
    uint32_t tlas_nodes, blas_nodes, triangles, instances;
    uint32_t max_depth;       /* deepest TLAS + BLAS node path (stack bound) */
    uint32_t node_bytes;      /* bytes per wide node */
    uint32_t triangle_bytes;  /* bytes per leaf triangle record */
} vvpt_bvh_info;
vvpt_status vvpt_get_bvh_info(const vvpt_ctx *ctx, vvpt_bvh_info *out);

/* ---------------------------------------------------------------- sampler -- */

/* The extended mode's sampler (no counterpart in the reference, which draws from one xorshift stream per pixel
 * and batch, rng_def.glsl:4-36): out[k * dims + d] = dimension d of sample first + k of the sequence of pixel
 * index `pixel` (y * width + x) under `seed`, computed on the GPU of ctx, or on the host when ctx is NULL; the two
 * are bit-identical.  count * dims <= 2^28. */
vvpt_status vvpt_sample_sequence(vvpt_ctx *ctx, uint32_t pixel, uint32_t seed, uint32_t first, uint32_t count,
                                 uint32_t dims, float *out);

/* ---------------------------------------------------------------- builders -- */

/* Acceleration-structure builder of vvpt_set_scene.  The reference leaves the build to the Vulkan driver
 * (vkCmdBuildAccelerationStructuresKHR, VulkanAccelerationStructure.cpp:137-140,258-259); both builders here make
 * the same two-level shape (one BLAS per mesh, a TLAS over the instances) of 8-wide compressed nodes. */
typedef enum {
    VVPT_BUILDER_SAH = 0, /* binned-SAH binary tree on the host, collapsed depth-first (default) */
    VVPT_BUILDER_LBVH = 1 /* linear BVH (Morton codes, radix sort, Karras hierarchy) on the GPU, collapsed
                             breadth-first; bit-exact with vvpt_build_lbvh(NULL, ...) */
} vvpt_builder;
/* Takes effect at the next vvpt_set_scene. */
vvpt_status vvpt_set_builder(vvpt_ctx *ctx, uint32_t builder);

typedef struct {
    uint32_t num_nodes;      /* wide nodes written (node 0 is the root) */
    uint32_t num_leaf_refs;  /* = n */
    uint32_t depth;          /* wide-node levels */
    double build_ms;         /* GPU: hipEvents around the build kernels (host <-> device copies excluded); host: wall time */
} vvpt_lbvh_info;

/* Stand-alone LBVH over n boxes (6 floats each: lo xyz, hi xyz), on the GPU of ctx, or on the host when ctx is
 * NULL.  Every output is a caller-owned host array and may be NULL:
 *   morton[n]       Morton codes in sorted order (10 bits per axis, x highest)
 *   order[n]        primitive index at each sorted position
 *   inner[2(n-1)]   left, right child of each binary internal node (0x80000000 | position for a leaf)
 *   nodes           wide nodes, 80 bytes each (vvpt_bvh_info.node_bytes), room for max(n, 1)
 *   leaf_refs[n]    primitive indices in leaf order
 * max_leaf (1..3) is the largest binary subtree that becomes one leaf child. */
vvpt_status vvpt_build_lbvh(vvpt_ctx *ctx, const float *boxes, uint32_t n, uint32_t max_leaf, uint32_t *morton,
                            uint32_t *order, uint32_t *inner, void *nodes, uint32_t *leaf_refs, vvpt_lbvh_info *info);

/* ------------------------------------------------- neural radiance cache -- */

/* The extended mode's learned radiance cache (no counterpart in the reference): 16-level hash-grid encoding of
 * the position plus spherical harmonics of the outgoing direction, roughness and albedo into an MLP of 5 hidden
 * layers of 64 ReLU units (bf16 weights on the matrix cores, fp32 accumulation), trained online with Adam on the
 * relative L2 loss.  The hooks below expose the cache's kernels for tests; an input is 10 floats: position xyz,
 * outgoing direction xyz, roughness, albedo rgb; a prediction or target is 3 floats (RGB radiance).  Batches hold
 * at most 65536 samples.  The cache of a context is created on first use. */
#define VVPT_NRC_INPUT_FLOATS 10u
#define VVPT_NRC_MLP_PARAMS 21504u                   /* 5 x 64 x 64 + 64 x 16, [layer][in][out] */
#define VVPT_NRC_GRID_PARAMS (16u * 524288u * 2u)    /* [level][entry][feature] */
/* (Re)initialise the weights and grid from `seed`; lo/hi (may be NULL) set the box positions are normalised to. */
vvpt_status vvpt_nrc_reset(vvpt_ctx *ctx, uint32_t seed, const float *lo, const float *hi);
vvpt_status vvpt_nrc_infer(vvpt_ctx *ctx, const float *inputs, uint32_t n, float *out);
/* `steps` Adam steps on one batch; losses[k] (may be NULL) receives the loss before step k. */
vvpt_status vvpt_nrc_train(vvpt_ctx *ctx, const float *inputs, const float *targets, uint32_t n, uint32_t steps,
                           float *losses);
/* Loss and gradients of one batch without an update (mlp_grad: VVPT_NRC_MLP_PARAMS floats, grid_grad:
 * VVPT_NRC_GRID_PARAMS floats; either may be NULL). */
vvpt_status vvpt_nrc_gradients(vvpt_ctx *ctx, const float *inputs, const float *targets, uint32_t n, float *loss,
                               float *mlp_grad, float *grid_grad);
/* Read (write = 0) or replace (write = 1) the fp32 master parameters; either array may be NULL. */
vvpt_status vvpt_nrc_params(vvpt_ctx *ctx, float *mlp, float *grid, int write);

#ifdef __cplusplus
}
#endif
#endif /* VVPT_H */
