/*
 * traverse.h - two-level wide-BVH traversal for gfx950.
 *
 * Replaces the driver traversal behind traceRayEXT (raygen.rgen.glsl:110,
 * lightSampling.glsl:128, next_event_estimation.glsl:21).  One lane walks one
 * ray; nodes are 80-byte compressed 8-wide nodes read with five dwordx4 loads.
 * The traversal stack holds node groups (child base index, remaining hit bits)
 * in LDS, one column per lane ([entry][lane] so a wave's accesses are
 * bank-conflict free).  Children are visited in the octant order set at build
 * time: the hit bit of internal child `slot` is 24 + (slot ^ oct_inv) and the
 * highest set bit is taken first, so no per-node sort is needed.
 *
 * Query modes:
 *   MODE_CLOSEST  closest hit in [tmin, tmax]
 *   MODE_CLOSEST2 two closest-hit answers in one walk: `hit` over [tmin2, tmax]
 *                 and `hitA` over [tmin, tmax] (tmin < tmin2), used to answer a
 *                 path ray (tmin 1e-3) and the BSDF-direction emitter lookup
 *                 (tmin 1e-4) that share origin and direction
 *   MODE_ANY      any hit in [tmin, tmax] (occlusion)
 *   MODE_ORDERED  closest hit after (prev_t, prev_key): one step of a
 *                 closest-first walk over all candidates, used to apply the
 *                 reference's any-hit logic in a deterministic order
 *   MODE_ANYHIT   every candidate in [tmin, tmax] goes to a callback that may
 *                 stop the walk (order-independent any-hit logic)
 * Equal distances resolve to the smaller (instance, primitive) key.
 */
#pragma once
#include "device_math.h"
#include "layout.h"

namespace vvpt {

/* One render job: its camera, acceleration-structure root, light list and render settings.  A single render
 * carries one in DScene::job (a kernel argument); a batch of jobs sharing one BVH pool keeps one per job in
 * device memory (DScene::jobs) and each path slot names its job. */
struct JobView {
    /* SceneData (core/Scene.hpp:27-35) of the job's scene part */
    float vi[16], pi[16];
    float lens, focal, znear, zfar;
    int32_t cam_volume;
    uint32_t tlas_root;
    uint32_t light_begin, num_lights; /* the part's lights in DScene::lights */
    uint32_t num_sel;                 /* lights a light sample chooses among: num_lights, +1 for a sampled environment */
    uint32_t scene_flags;             /* SCENE_HAS_* of the job's scene part */
    /* RenderInfo of the job */
    uint32_t W, H, npix;
    uint32_t batch_size, batch_begin, depth, seed;
    float total_samples;
    uint32_t item_begin, items;       /* the job's work items (pixel, batch) in the launch */
    uint32_t *remaining;              /* batch: items not yet finished */
    unsigned long long *done_ticks;   /* batch: wall clock when the job's last item finished */
};

struct DScene {
    const WideNode *nodes;
    const LeafTri *tris;
    const TlasLeaf *tlas_leaf;
    const DInstance *insts;
    const DVertex *tri_verts; /* the three vertices of every triangle, in global triangle order */
    const DMaterial *mats;
    const DMaterial *inst_mats; /* each instance's material, in instance order */
    const DTexture *texs;
    const uint32_t *tex8;
    const float4 *texf;
    const DLight *lights;
    const float4 *cube;
    const float *srgb_lut;
    uint32_t cube_w;
    uint32_t scene_flags; /* union over the scene parts of bit0: some material is transparent, bit1: some
                           * instance changes volume (per-part flags in JobView) */
    uint32_t env_type;
    float bg[3];
    float env_intensity;
    float flat_normal[3]; /* texel of the default normal map */
    JobView job;          /* the render job (single render) */
    const JobView *jobs;  /* the jobs of a batch (batched render), else null */
    uint32_t njobs;
    /* extended mode */
    uint32_t env_mw, env_mh;    /* environment importance grid (0 when absent) */
    const float *env_prob;      /* alias table: acceptance of each cell */
    const uint32_t *env_alias;  /* alias table: the other cell */
    const float *env_cpdf;      /* probability of each cell */
};

enum : uint32_t { SCENE_HAS_TRANSPARENT = 1u, SCENE_HAS_VOLUME_CHANGE = 2u };

struct TraceHit {
    float t, u, v;
    uint32_t inst, prim;
};

struct TraceCount {
    uint32_t nodes, tris;
};

enum { MODE_CLOSEST = 0, MODE_CLOSEST2 = 1, MODE_ANY = 2, MODE_ORDERED = 3, MODE_ANYHIT = 4 };

__device__ __forceinline__ bool key_less(uint32_t ia, uint32_t pa, uint32_t ib, uint32_t pb) {
    return ia < ib || (ia == ib && pa < pb);
}

/* Reciprocal direction for the slab tests.  The hardware reciprocal (1 ulp) is enough: the node test accepts a child
 * when tn <= tf * 1.000001, a margin of about 8 ulp, so no box the exact reciprocal would accept is rejected; the
 * triangle test, whose results are the query's output, divides exactly. */
__device__ __forceinline__ float safe_inv(float x) { return x == 0.0f ? copysignf(1e30f, x) : __builtin_amdgcn_rcpf(x); }

__device__ __forceinline__ uint32_t octant_inv(f3 d) {
    uint32_t o = (d.x < 0.0f ? 1u : 0u) | (d.y < 0.0f ? 2u : 0u) | (d.z < 0.0f ? 4u : 0u);
    return o ^ 7u;
}

/* Slab test of the 8 children of node `idx`; returns the hit mask
 * (internal children in bits 24..31 after the octant xor, leaf primitives in
 * bits 0..23) and the node's child/leaf bases and internal-child mask. */
__device__ __forceinline__ uint32_t intersect_node(const WideNode *__restrict__ nodes, uint32_t idx, f3 O, f3 idir,
                                                   uint32_t oct_inv, float tmin, float tmax, uint32_t &child_base,
                                                   uint32_t &leaf_base, uint32_t &imask) {
    const uint4 *p = reinterpret_cast<const uint4 *>(nodes + idx);
    const uint4 w0 = p[0];
    const uint4 w1 = p[1];
    const uint4 w2 = p[2];
    const uint4 w3 = p[3];
    const uint4 w4 = p[4];
    const uint32_t ei = w0.w;
    const float sx = __uint_as_float((ei & 0xffu) << 23);
    const float sy = __uint_as_float(((ei >> 8) & 0xffu) << 23);
    const float sz = __uint_as_float(((ei >> 16) & 0xffu) << 23);
    imask = ei >> 24;
    child_base = w1.x;
    leaf_base = w1.y;
    const float ax = sx * idir.x, ay = sy * idir.y, az = sz * idir.z;
    const float bx = (__uint_as_float(w0.x) - O.x) * idir.x;
    const float by = (__uint_as_float(w0.y) - O.y) * idir.y;
    const float bz = (__uint_as_float(w0.z) - O.z) * idir.z;
    const bool nx = idir.x < 0.0f, ny = idir.y < 0.0f, nz = idir.z < 0.0f;
    uint32_t hitmask = 0;
    const uint32_t octx4 = oct_inv * 0x01010101u;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
        uint32_t meta4 = half ? w1.w : w1.z;
        /* an internal child (meta 001 11sss) takes bit 24 + (s ^ oct_inv): bit 4 of its meta byte and bit 3 are
         * set, which no leaf offset (< 24) or empty slot (0) has; one byte-parallel xor serves 4 children */
        const uint32_t inner4 = meta4 & (meta4 << 1) & 0x10101010u;
        meta4 ^= (inner4 - (inner4 >> 4)) & octx4;
        const uint32_t lox = half ? w2.y : w2.x, loy = half ? w2.w : w2.z, loz = half ? w3.y : w3.x;
        const uint32_t hix = half ? w3.w : w3.z, hiy = half ? w4.y : w4.x, hiz = half ? w4.w : w4.z;
        const uint32_t nearx = nx ? hix : lox, farx = nx ? lox : hix;
        const uint32_t neary = ny ? hiy : loy, fary = ny ? loy : hiy;
        const uint32_t nearz = nz ? hiz : loz, farz = nz ? loz : hiz;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t sh = 8 * j;
            const float tnx = fmaf((float)((nearx >> sh) & 0xffu), ax, bx);
            const float tny = fmaf((float)((neary >> sh) & 0xffu), ay, by);
            const float tnz = fmaf((float)((nearz >> sh) & 0xffu), az, bz);
            const float tfx = fmaf((float)((farx >> sh) & 0xffu), ax, bx);
            const float tfy = fmaf((float)((fary >> sh) & 0xffu), ay, by);
            const float tfz = fmaf((float)((farz >> sh) & 0xffu), az, bz);
            const float tn = fmaxf(fmaxf(tnx, tny), fmaxf(tnz, tmin));
            const float tf = fminf(fminf(tfx, tfy), fminf(tfz, tmax));
            /* (meta >> 5) << (meta & 31): the unary triangle count at the leaf offset, or one bit for an internal
             * child; an empty slot (meta 0) adds nothing */
            const uint32_t bits = ((meta4 >> (sh + 5)) & 7u) << ((meta4 >> sh) & 0x1fu);
            if (tn <= tf * 1.000001f) hitmask |= bits;
        }
    }
    return hitmask;
}

/* Moller-Trumbore with the explicit fma order of the CPU restatement.  A
 * division-free pre-test rejects most misses first; it only rejects when the
 * exact test below would also reject (its margins are far wider than the
 * rounding of the divided values), so accepted hits are bit-identical. */
__device__ __forceinline__ bool intersect_tri(f3 o, f3 d, const LeafTri *__restrict__ tris, uint32_t idx, float tmax,
                                              float &t, float &u, float &v, uint32_t &prim) {
    const float4 *p = reinterpret_cast<const float4 *>(tris + idx);
    const float4 a = p[0], b = p[1], c = p[2];
    const f3 e1 = {b.x, b.y, b.z}, e2 = {c.x, c.y, c.z};
    const f3 pv = fcross(d, e2);
    const float det = fdot(e1, pv);
    if (det == 0.0f) return false;
    const f3 s = {o.x - a.x, o.y - a.y, o.z - a.z};
    const float un = fdot(s, pv);
    const f3 q = fcross(s, e1);
    const float vn = fdot(d, q);
    const float tn = fdot(e2, q);
    /* pre-test on the undivided values: x = n / det is outside [lo, hi] beyond doubt */
    const float ad = fabsf(det), sg = det < 0.0f ? -1.0f : 1.0f;
    const float slack = ad * 1e-5f;
    if (un * sg < -slack || vn * sg < -slack || (un + vn) * sg > ad + slack) return false;
    if (tn * sg > tmax * ad * 1.0001f + slack) return false;
    const float inv = 1.0f / det;
    u = un * inv;
    if (!(u >= 0.0f && u <= 1.0f)) return false;
    v = vn * inv;
    if (!(v >= 0.0f && u + v <= 1.0f)) return false;
    t = tn * inv;
    prim = __float_as_uint(a.w);
    return true;
}

/* No-op any-hit callback for the modes that do not need one. */
struct NoAnyHit {
    __device__ __forceinline__ bool operator()(const TraceHit &) { return false; }
};

/*
 * Walk the two-level BVH.  `st` is this lane's LDS stack column (entries at
 * st[k * BLOCK]).  Returns true if anything was accepted.  MODE_ANYHIT calls
 * anyhit(candidate) for every hit in [tmin, tmax] (in traversal order) and
 * stops when it returns true.
 *
 * Loop structure: an inner node loop runs until the lane has a leaf group to
 * test (or is done), then an inner leaf loop tests that group, so a wave's
 * lanes mostly run node steps together and leaf steps together.
 */
template <int MODE, int STACK, int BLOCK, bool COUNT, class AnyHit = NoAnyHit>
__device__ __forceinline__ bool trace_ray(const DScene &S, const uint32_t root, const f3 O, const f3 D, const float tmin,
                                          const float tmax,
                                          TraceHit &hit, TraceHit &hitA, const float tmin2, const float prev_t,
                                          const uint32_t prev_inst, const uint32_t prev_prim, uint2 *st,
                                          TraceCount &cnt, AnyHit *anyhit = nullptr) {
    hit.t = tmax;
    hit.inst = kInvalid;
    hit.prim = kInvalid;
    hit.u = hit.v = 0.0f;
    if (MODE == MODE_CLOSEST2) {
        hitA = hit;
    }
    const float tlo = (MODE == MODE_ORDERED) ? fmaxf(tmin, prev_t) : tmin;

    f3 ro = O, rd = D;
    f3 idir = {safe_inv(D.x), safe_inv(D.y), safe_inv(D.z)};
    uint32_t oct_inv = octant_inv(D);

    uint2 ng = make_uint2(root, 0x80000000u); /* virtual group holding the root */
    uint2 tg = make_uint2(0u, 0u);
    int sp = 0;
    bool in_blas = false;
    uint32_t cur_inst = 0;
    uint2 saved_ng = make_uint2(0u, 0u), saved_tg = make_uint2(0u, 0u);
    int blas_sp = 0;
    bool found = false;

    for (;;) {
        /* ---- node phase: descend until a leaf group is pending ---- */
        while (tg.y == 0u) {
            if (ng.y > 0x00ffffffu) {
                const uint32_t bit = 31u - __builtin_clz(ng.y);
                ng.y &= ~(1u << bit);
                const uint32_t slot = (bit - 24u) ^ oct_inv;
                const uint32_t rel = __builtin_popcount(ng.y & 0xffu & ((1u << slot) - 1u));
                const uint32_t node = ng.x + rel;
                if (ng.y > 0x00ffffffu && sp < STACK) {
                    st[sp * BLOCK] = ng;
                    ++sp;
                }
                const float tcull = (MODE == MODE_ANY || MODE == MODE_ANYHIT) ? tmax : hit.t;
                uint32_t cb, lb, im;
                if (COUNT) cnt.nodes++;
                const uint32_t hm = intersect_node(S.nodes, node, ro, idir, oct_inv, tlo, tcull, cb, lb, im);
                ng = make_uint2(cb, (hm & 0xff000000u) | im);
                tg = make_uint2(lb, hm & 0x00ffffffu);
            } else if (in_blas && sp == blas_sp) {
                in_blas = false;
                ro = O;
                rd = D;
                idir = {safe_inv(D.x), safe_inv(D.y), safe_inv(D.z)};
                oct_inv = octant_inv(D);
                ng = saved_ng;
                tg = saved_tg;
            } else if (sp == 0) {
                return found;
            } else {
                --sp;
                ng = st[sp * BLOCK];
            }
        }
        /* ---- leaf phase ---- */
        if (!in_blas) {
            /* TLAS leaf: enter the instance's BLAS in object space */
            const uint32_t bit = __builtin_ctz(tg.y);
            tg.y &= tg.y - 1u;
            const float4 *w = reinterpret_cast<const float4 *>(S.tlas_leaf + tg.x + bit);
            const float4 r0 = w[0], r1 = w[1], r2 = w[2];
            const uint4 lf = reinterpret_cast<const uint4 *>(w)[3];
            cur_inst = lf.x;
            const float m[12] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w, r2.x, r2.y, r2.z, r2.w};
            ro = xform_point(m, O);
            rd = xform_vector(m, D);
            idir = {safe_inv(rd.x), safe_inv(rd.y), safe_inv(rd.z)};
            oct_inv = octant_inv(rd);
            saved_ng = ng;
            saved_tg = tg;
            blas_sp = sp;
            in_blas = true;
            ng = make_uint2(lf.y, 0x80000000u);
            tg.y = 0u;
            continue;
        }
        while (tg.y != 0u) {
            const uint32_t bit = __builtin_ctz(tg.y);
            tg.y &= tg.y - 1u;
            const uint32_t idx = tg.x + bit;
            float t, u, v;
            uint32_t prim;
            if (COUNT) cnt.tris++;
            const float tcull = (MODE == MODE_ANY || MODE == MODE_ANYHIT) ? tmax : hit.t;
            if (intersect_tri(ro, rd, S.tris, idx, tcull, t, u, v, prim)) {
                if (MODE == MODE_ANY) {
                    if (t >= tmin && t <= tmax) {
                        hit = {t, u, v, cur_inst, prim};
                        return true;
                    }
                } else if (MODE == MODE_ANYHIT) {
                    if (t >= tmin && t <= tmax) {
                        const TraceHit cand = {t, u, v, cur_inst, prim};
                        found = true;
                        if ((*anyhit)(cand)) {
                            hit = cand;
                            return true;
                        }
                    }
                } else if (MODE == MODE_CLOSEST2) {
                    if (t >= tmin && (t < hitA.t || (t == hitA.t && key_less(cur_inst, prim, hitA.inst, hitA.prim)))) {
                        hitA = {t, u, v, cur_inst, prim};
                        found = true;
                    }
                    if (t >= tmin2 && (t < hit.t || (t == hit.t && key_less(cur_inst, prim, hit.inst, hit.prim)))) {
                        hit = {t, u, v, cur_inst, prim};
                        found = true;
                    }
                } else {
                    bool ok = t >= tmin && (t < hit.t || (t == hit.t && key_less(cur_inst, prim, hit.inst, hit.prim)));
                    if (MODE == MODE_ORDERED)
                        ok = ok && (t > prev_t || (t == prev_t && key_less(prev_inst, prev_prim, cur_inst, prim)));
                    if (ok) {
                        hit = {t, u, v, cur_inst, prim};
                        found = true;
                    }
                }
            }
        }
    }
}

/*
 * Restartable traversal for persistent kernels: the walk state lives in
 * registers, step() advances one node phase plus one leaf phase and reports
 * when the ray is finished, so a lane whose ray ends can take a new ray while
 * the rest of its wave keeps walking (lanes otherwise idle until the longest
 * ray of the wave ends).  Modes: MODE_CLOSEST2 (tmin2 == tmin gives a plain
 * closest-hit query), MODE_ANY and MODE_ANYHIT.
 */
/* Walk state of one lane (registers).  The world-space ray, needed only when the walk enters or leaves an instance,
 * lives in three extra LDS entries of the lane's stack (entries STACK .. STACK + 2), which keeps the persistent trace
 * kernels within the registers of 5 waves per SIMD. */
struct Trav {
    f3 ro, rd, idir;
    uint32_t oct_inv;
    uint2 ng, tg;
    int sp, blas_sp; /* inside a BLAS, entries blas_sp - 2 and blas_sp - 1 hold the TLAS walk's ng and tg */
    bool in_blas;
    bool cur_pass; /* current instance is passed by emitter lookups (INST_NEE_PASS) */
    uint32_t cur_inst;
    float tmin, tmin2, tmax;
    float tskip;   /* MODE_CLOSEST2: nearest passed candidate at or beyond tmin */
    TraceHit hit, hitA;
};

/* MODE_CLOSEST2 answers two queries in one walk: `hit` = closest candidate in
 * [tmin2, tmax] (the path ray), `hitA` = closest candidate in [tmin, tmaxA]
 * that is not passed by emitter lookups (the first surface that can stop a
 * BSDF-direction lookup, next_event_estimation.glsl with rayNEE.rahit.glsl);
 * `tskip` records the nearest passed candidate so the caller knows whether the
 * 1 - alpha product of the passed surfaces before hitA is needed. */
template <int STACK, int BLOCK>
__device__ __forceinline__ void ray_store(uint2 *st, f3 O, f3 D) {
    st[STACK * BLOCK] = make_uint2(__float_as_uint(O.x), __float_as_uint(O.y));
    st[(STACK + 1) * BLOCK] = make_uint2(__float_as_uint(O.z), __float_as_uint(D.x));
    st[(STACK + 2) * BLOCK] = make_uint2(__float_as_uint(D.y), __float_as_uint(D.z));
}
template <int STACK, int BLOCK>
__device__ __forceinline__ void ray_load(const uint2 *st, f3 &O, f3 &D) {
    const uint2 a = st[STACK * BLOCK], b = st[(STACK + 1) * BLOCK], c = st[(STACK + 2) * BLOCK];
    O = {__uint_as_float(a.x), __uint_as_float(a.y), __uint_as_float(b.x)};
    D = {__uint_as_float(b.y), __uint_as_float(c.x), __uint_as_float(c.y)};
}

template <int STACK, int BLOCK>
__device__ __forceinline__ void trav_init(Trav &w, uint2 *st, uint32_t root, f3 O, f3 D, float tmin, float tmin2,
                                          float tmax, float tmaxA = 0.0f) {
    ray_store<STACK, BLOCK>(st, O, D);
    w.ro = O;
    w.rd = D;
    w.idir = {safe_inv(D.x), safe_inv(D.y), safe_inv(D.z)};
    w.oct_inv = octant_inv(D);
    w.ng = make_uint2(root, 0x80000000u);
    w.tg = make_uint2(0u, 0u);
    w.sp = 0;
    w.blas_sp = 0;
    w.in_blas = false;
    w.cur_inst = 0;
    w.tmin = tmin;
    w.tmin2 = tmin2;
    w.tmax = tmax;
    w.hit = {tmax, 0.0f, 0.0f, kInvalid, kInvalid};
    w.hitA = {tmaxA > 0.0f ? fminf(tmaxA, tmax) : tmax, 0.0f, 0.0f, kInvalid, kInvalid};
    w.tskip = 3.0e38f;
    w.cur_pass = false;
}

/* Returns true when the walk is over (for MODE_ANY/MODE_ANYHIT: also when stopped on a hit).  One call does one
 * unit of work per lane - one triangle test, one node test (after the pops, instance entry or exit that lead to it),
 * or the last triangle test of a leaf group followed by the next node test - so the lanes of a wave stay busy: a
 * call that ran a lane's node loop or leaf loop to its end would hold every other lane of the wave until the
 * slowest lane found its next leaf.  The order in which one ray
 * visits nodes and triangles is that of the recursive walk, whatever the interleaving of the wave's lanes. */
template <int MODE, int STACK, int BLOCK, bool COUNT, class AnyHit = NoAnyHit>
__device__ __forceinline__ bool trav_step(Trav &w, const DScene &S, uint2 *st, TraceCount &cnt,
                                          AnyHit *anyhit = nullptr) {
    if (w.tg.y != 0u && w.in_blas) {
        /* ---- kTrisPerStep triangles of the current leaf group per call.  Measured on the 1080p field with the
         * SAH-collapsed BVH (3 triangle tests per ray): 1 per call 749, 2 730, 3 705 Msamples/s; a second test
         * in the same call mostly runs with the lanes that have no second triangle idle ---- */
        constexpr int kTrisPerStep = 1;
        for (int k = 0; k < kTrisPerStep; ++k) {
            if (w.tg.y == 0u) break;
            const uint32_t bit = __builtin_ctz(w.tg.y);
            w.tg.y &= w.tg.y - 1u;
            const uint32_t idx = w.tg.x + bit;
            float t, u, v;
            uint32_t prim;
            if (COUNT) cnt.tris++;
            const float tcull = (MODE == MODE_CLOSEST2) ? fmaxf(w.hit.t, w.hitA.t) : w.tmax;
            if (intersect_tri(w.ro, w.rd, S.tris, idx, tcull, t, u, v, prim)) {
                if (MODE == MODE_ANY) {
                    if (t >= w.tmin && t <= w.tmax) {
                        w.hit = {t, u, v, w.cur_inst, prim};
                        return true;
                    }
                } else if (MODE == MODE_ANYHIT) {
                    if (t >= w.tmin && t <= w.tmax) {
                        const TraceHit cand = {t, u, v, w.cur_inst, prim};
                        if ((*anyhit)(cand)) {
                            w.hit = cand;
                            return true;
                        }
                    }
                } else {
                    if (t >= w.tmin) {
                        if (w.cur_pass)
                            w.tskip = fminf(w.tskip, t);
                        else if (t < w.hitA.t || (t == w.hitA.t && key_less(w.cur_inst, prim, w.hitA.inst, w.hitA.prim)))
                            w.hitA = {t, u, v, w.cur_inst, prim};
                    }
                    if (t >= w.tmin2 &&
                        (t < w.hit.t || (t == w.hit.t && key_less(w.cur_inst, prim, w.hit.inst, w.hit.prim))))
                        w.hit = {t, u, v, w.cur_inst, prim};
                }
            }
        }
        /* a lane whose leaf group is used up goes on to its next node in the same call: the wave runs that node
         * test for its other lanes anyway, and this lane would otherwise sit it out */
        if (w.tg.y != 0u) return false;
    } else if (w.tg.y != 0u) {
        /* ---- TLAS leaf: enter the next instance's BLAS ---- */
        const uint32_t bit = __builtin_ctz(w.tg.y);
        w.tg.y &= w.tg.y - 1u;
        const float4 *q = reinterpret_cast<const float4 *>(S.tlas_leaf + w.tg.x + bit);
        const float4 r0 = q[0], r1 = q[1], r2 = q[2];
        const uint4 lf = reinterpret_cast<const uint4 *>(q)[3];
        w.cur_inst = lf.x;
        if (MODE == MODE_CLOSEST2) w.cur_pass = (lf.z & INST_NEE_PASS) != 0u;
        const float m[12] = {r0.x, r0.y, r0.z, r0.w, r1.x, r1.y, r1.z, r1.w, r2.x, r2.y, r2.z, r2.w};
        f3 O, D;
        ray_load<STACK, BLOCK>(st, O, D);
        w.ro = xform_point(m, O);
        w.rd = xform_vector(m, D);
        w.idir = {safe_inv(w.rd.x), safe_inv(w.rd.y), safe_inv(w.rd.z)};
        w.oct_inv = octant_inv(w.rd);
        /* the TLAS position goes on the stack under the BLAS walk's entries */
        st[w.sp * BLOCK] = w.ng;
        st[(w.sp + 1) * BLOCK] = w.tg;
        w.sp += 2;
        w.blas_sp = w.sp;
        w.in_blas = true;
        w.ng = make_uint2(lf.y, 0x80000000u);
        w.tg.y = 0u;
    }
    /* ---- pops and instance exits up to the next node to test ---- */
    while (w.ng.y <= 0x00ffffffu) {
        if (w.in_blas && w.sp == w.blas_sp) {
            w.in_blas = false;
            f3 O, D;
            ray_load<STACK, BLOCK>(st, O, D);
            w.ro = O;
            w.rd = D;
            w.idir = {safe_inv(D.x), safe_inv(D.y), safe_inv(D.z)};
            w.oct_inv = octant_inv(D);
            w.sp -= 2;
            w.ng = st[w.sp * BLOCK];
            w.tg = st[(w.sp + 1) * BLOCK];
            if (w.tg.y != 0u) return false; /* more instances of the same TLAS leaf group first */
        } else if (w.sp == 0) {
            return true;
        } else {
            --w.sp;
            w.ng = st[w.sp * BLOCK];
        }
    }
    /* ---- one node ---- */
    const uint32_t bit = 31u - __builtin_clz(w.ng.y);
    w.ng.y &= ~(1u << bit);
    const uint32_t slot = (bit - 24u) ^ w.oct_inv;
    const uint32_t rel = __builtin_popcount(w.ng.y & 0xffu & ((1u << slot) - 1u));
    const uint32_t node = w.ng.x + rel;
    if (w.ng.y > 0x00ffffffu && w.sp < STACK) {
        st[w.sp * BLOCK] = w.ng;
        ++w.sp;
    }
    const float tcull = (MODE == MODE_CLOSEST2) ? fmaxf(w.hit.t, w.hitA.t) : w.tmax;
    uint32_t cb, lb, im;
    if (COUNT) cnt.nodes++;
    const uint32_t hm = intersect_node(S.nodes, node, w.ro, w.idir, w.oct_inv, w.tmin, tcull, cb, lb, im);
    w.ng = make_uint2(cb, (hm & 0xff000000u) | im);
    w.tg = make_uint2(lb, hm & 0x00ffffffu);
    return false;
}

}  // namespace vvpt
