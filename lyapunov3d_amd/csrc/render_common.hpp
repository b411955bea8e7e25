/*
 * render_common.hpp - what the render's kernels share: the launch table's
 * entries, vectors, shading, the box clip, lambda in the coefficient window,
 * the output records and the lists of rays between launches.
 */
#pragma once

#include "internal.hpp"
#include "lists.hpp"

namespace lyap {

/* One view of a render launch, in device memory. */
struct ViewDesc {
    EvalDesc e;
    LyapCam cam;
    LyapParams prm;
    uint32_t w, h;
    uint32_t blocks_x;         /* 8x8 pixel blocks per row */
    uint32_t n_rays;           /* 64 * blocks, padded past the image edge */
    uint32_t tile_begin;       /* first tile of this view in the launch */
    uint32_t n_tiles;
    LyapRGBA *rgba;
    LyapPoint *points;
    float *depth;
    float *lambda;
    uint32_t *evals;
    const LyapLight *lights;
    uint32_t num_lights;
    int32_t refine;            /* LYAP_REFINE_* */
    int32_t bisect_steps;
    float normal_h;
    float margin;              /* FP64 re-evaluation margin during bisection */
    uint32_t max_samples;
    uint32_t ray_begin;        /* first ray of this launch (a view may be split) */
    uint32_t cont_base;        /* this view's region of the continuation buffers */
    uint32_t cont_cap;
    uint32_t refine_base;      /* this view's region of the refinement records */
    uint32_t refine_cap;       /* records per sub-list */
    uint32_t ray_base;         /* first ray of this view in a grid of one lane per ray */
    uint32_t tile_len;         /* rays per level-0 work-queue tile */
};

/* Words between counters that different waves update: one 128-byte line. */
constexpr uint32_t kHeadStride = 32;

/* A ray whose march found its opaque sample, waiting for the refinement
 * launch: the bisection interval [lo, hi] with lambda at both ends, the
 * march step (the normal offset of the reference's method), the march sums
 * and the evaluations so far (48 bytes). */
struct alignas(16) RefineRec {
    uint32_t pix, evals;
    float Vx, Vy, Vz, lo, hi, l_hi, dt, a, c, l_lo;
};
static_assert(sizeof(RefineRec) == 48, "refinement record size");

/* The refinement records of a view are kept in sub-lists with a counter each
 * on a 128-byte line, taken by block index: waves of one XCD share a counter
 * (device-scope atomics on a line that waves of several XCDs update are
 * slow). The persistent levels use kRefineSubs, the march passes
 * MarchPlan::subs for these and for the rays they list. */
constexpr uint32_t kRefineSubs = 8;

struct F3 { float x, y, z; };
__device__ __forceinline__ F3 f3(const LyapVec &v) { return {v.x, v.y, v.z}; }
__device__ __forceinline__ F3 add(F3 a, F3 b) { return {a.x + b.x, a.y + b.y, a.z + b.z}; }
__device__ __forceinline__ F3 sub(F3 a, F3 b) { return {a.x - b.x, a.y - b.y, a.z - b.z}; }
__device__ __forceinline__ F3 mul(F3 a, float s) { return {a.x * s, a.y * s, a.z * s}; }
__device__ __forceinline__ F3 divv(F3 a, float s) { return {a.x / s, a.y / s, a.z / s}; }
__device__ __forceinline__ float dot(F3 a, F3 b) { return a.x * b.x + a.y * b.y + a.z * b.z; }
__device__ __forceinline__ float mag2(F3 a) { return a.x * a.x + a.y * a.y + a.z * a.z; }
/* Vec::normalize (vec3.hpp:141-154) */
__device__ __forceinline__ F3 normalized(F3 a)
{
    const float m2 = mag2(a);
    if ((double)m2 < 1e-12) return {0.f, 0.f, 0.f};
    if (m2 == 1.0f) return a;
    return divv(a, sqrtf(m2));
}
__device__ __forceinline__ float clamp01(float v) { return v < 0.0f ? 0.0f : (v > 1.0f ? 1.0f : v); }

struct C4 { float x, y, z, w; };
__device__ __forceinline__ C4 col(const LyapColor &c) { return {c.x, c.y, c.z, c.w}; }
__device__ __forceinline__ C4 cadd(C4 a, C4 b) { return {a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w}; }
__device__ __forceinline__ C4 cmul(C4 a, float s) { return {a.x * s, a.y * s, a.z * s, a.w * s}; }

/* shade (kernel.cu:25-106) */
__device__ inline C4 shade(F3 P, F3 N, float a, float c, const LyapCam &cam,
                    const LyapLight *lights, uint32_t n_lights)
{
    C4 color = {0.f, 0.f, 0.f, 0.f};
    if (__builtin_isnan(a)) return color;
    const F3 camC = f3(cam.C);
    for (uint32_t li = 0; li < n_lights; ++li) {
        const LyapLight &L = lights[li];
        const F3 camV = sub(camC, P);
        F3 lightV = sub(f3(L.C), P);
        const float d2 = mag2(lightV);
        lightV = normalized(lightV);
        float i = dot(lightV, N);
        const float j = -dot(lightV, f3(L.V));
        C4 phong;
        if (j > L.lightOuterCone) {
            i = clamp01(i);
            const C4 diffuse = cmul(col(L.diffuseColor), i * L.diffusePower);
            const F3 halfV = normalized(add(camV, lightV));
            float s = clamp01(dot(N, halfV));
            s = powf(s, L.specularHardness);
            const C4 specular = cmul(col(L.specularColor), s * L.specularPower);
            phong = cmul(cadd(specular, diffuse), L.lightRange / d2);
            if (j < L.lightInnerCone)
                phong = cmul(phong, (j - L.lightOuterCone) / (L.lightInnerCone - L.lightOuterCone));
            phong = cadd(phong, col(L.ambient));
        } else {
            phong = col(L.ambient);
        }
        if (c > 0.0f) {
            const float k = (float)(0.1125 / (double)logf(c));
            phong = cadd(phong, cmul(col(L.chaosColor), k));
        }
        color = cadd(color, phong);
    }
    return color;
}

/* to_rgba (color.hpp:169-175), saturating. */
__device__ __forceinline__ unsigned char to_u8(float x)
{
    const double v = 255.0 * (double)x;
    if (!(v > 0.0)) return 0;
    if (v >= 255.0) return 255;
    return (unsigned char)v;
}

/* Box entry and exit (kernel.cu:181-285), plane parameters formed in double
 * and stored as float like the reference's double literals make them. */
__device__ inline bool clip_box(F3 C, F3 V, float lo, float hi, float &t0_out, float &t1_out)
{
    const double dlo = lo, dhi = hi;
    float ts[6];
    const float Ca[3] = {C.x, C.y, C.z};
    const float Va[3] = {V.x, V.y, V.z};
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        ts[2 * a] = (Va[a] != 0.0f) ? (float)((dlo - (double)Ca[a]) / (double)Va[a]) : INFINITY;
        ts[2 * a + 1] = (Va[a] != 0.0f) ? (float)((dhi - (double)Ca[a]) / (double)Va[a]) : INFINITY;
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        if (ts[k] == INFINITY) continue;
        const F3 P = add(C, mul(V, ts[k]));
        const float Pa[3] = {P.x, P.y, P.z};
        const int ax = k / 2;
        bool out = false;
#pragma unroll
        for (int b = 0; b < 3; ++b) {
            if (b == ax) continue;
            if ((double)Pa[b] < dlo || (double)Pa[b] > dhi) out = true;
        }
        if (out) ts[k] = NAN;
    }
    float t0 = 3.40282347e+38F, t1 = 0.0f;
    int i0 = -1, i1 = -1;
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        if (!__builtin_isfinite(ts[k])) continue;
        if (i0 == -1 || ts[k] < t0) { t0 = ts[k]; i0 = k; }
        if (i1 == -1 || ts[k] > t1) { t1 = ts[k]; i1 = k; }
    }
    if (i0 == -1 && i1 == -1) return false;
    if (i1 == -1 || i0 == i1) { t1 = t0; t0 = 0.0f; }
    if (t0 < 0) t0 = 0.0f;
    t0_out = t0;
    t1_out = t1;
    return true;
}

/* ---- lambda in the kernel's window ------------------------------------- */

template <int W>
__device__ __noinline__ float eval_fp64_call(const EvalDesc &e, float x, float y, float z)
{
    return (float)lambda_fp64_w<W>(x, y, z, e);
}

template <int W, int PREC>
__device__ __forceinline__ float eval_lambda(const EvalDesc &e, float x, float y, float z)
{
    if (PREC == LYAP_PREC_FP64) return (float)lambda_fp64_w<W>(x, y, z, e);
    if (PREC == LYAP_PREC_PLAIN) return lambda_plain_w<W>(x, y, z, e);
    return lambda_product_w<W>(x, y, z, e);
}

/* The view's output pointers, read together (one wait for all of them
 * rather than one per optional output). */
struct OutPtrs {
    LyapRGBA *rgba;
    LyapPoint *points;
    float *depth;
    float *lambda;
    uint32_t *evals;
    uint32_t present;      /* bit 0 points, 1 depth, 2 lambda, 3 evals */
};

__device__ __forceinline__ OutPtrs out_ptrs(const ViewDesc &v)
{
    OutPtrs o;
    o.rgba = v.rgba;
    o.points = v.points;
    o.depth = v.depth;
    o.lambda = v.lambda;
    o.evals = v.evals;
    o.present = (o.points ? 1u : 0u) | (o.depth ? 2u : 0u) | (o.lambda ? 4u : 0u) |
                (o.evals ? 8u : 0u);
    return o;
}

__device__ __forceinline__ void write_miss(const ViewDesc &v, uint32_t pix, uint32_t evals)
{
    const OutPtrs o = out_ptrs(v);
    if (o.present & 1u) {
        LyapPoint p;
        p.P = {0.f, 0.f, 0.f};
        p.N = {0.f, 0.f, 0.f};
        p.a = NAN;
        p.c = 0.f;
        p.l = NAN;
        o.points[pix] = p;
    }
    if (o.present & 2u) o.depth[pix] = NAN;
    if (o.present & 4u) o.lambda[pix] = NAN;
    if (o.present & 8u) o.evals[pix] = evals;
    LyapRGBA z = {0, 0, 0, 0};
    o.rgba[pix] = z;
}

/* A NaN normal component (a normal sample's lambda was NaN) as the one
 * quiet NaN: the refinement launch and refinement in place form the
 * differences in orders that agree on every number but not on a NaN's sign
 * bit. */
__device__ __forceinline__ float canonical(float x) { return __builtin_isnan(x) ? NAN : x; }

__device__ __forceinline__ void write_hit(const ViewDesc &v, uint32_t pix, uint32_t evals, F3 P, F3 N,
                                          float t, float l, float a, float c)
{
    const OutPtrs o = out_ptrs(v);
    if (o.present & 1u) {
        LyapPoint p;
        p.P = {P.x, P.y, P.z};
        p.N = {canonical(N.x), canonical(N.y), canonical(N.z)};
        p.a = a;
        p.c = c;
        p.l = l;
        o.points[pix] = p;
    }
    if (o.present & 2u) o.depth[pix] = t;
    if (o.present & 4u) o.lambda[pix] = l;
    if (o.present & 8u) o.evals[pix] = evals;
}

enum : int { RAY_PAD = 0, RAY_MISS = 1, RAY_HIT = 2 };

/* Pixel, direction and box interval of ray `id` of view v (pixel mapping
 * kernel.cu:500-516, direction :160-163, box clip :180-279). RAY_PAD for a
 * padding ray past the image edge. */
__device__ __forceinline__ int ray_setup(const ViewDesc &v, uint32_t id, uint32_t &pix, F3 &V,
                                         float &t0, float &t1)
{
    id += v.ray_begin;
    const uint32_t blk = id >> 6, in = id & 63u;
    const uint32_t px = (blk % v.blocks_x) * 8u + (in & 7u);
    const uint32_t py = (blk / v.blocks_x) * 8u + (in >> 3);
    if (px >= v.w || py >= v.h) return RAY_PAD;
    pix = px + py * v.w;
    V = add(add(f3(v.cam.S0), mul(f3(v.cam.SDX), (float)px)), mul(f3(v.cam.SDY), (float)py));
    V = normalized(V);
    V = divv(V, v.cam.M);
    return clip_box(f3(v.cam.C), V, v.prm.lMin, v.prm.lMax, t0, t1) ? RAY_HIT : RAY_MISS;
}
__device__ __forceinline__ void wave_sync_lds()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

/* Adds the lanes' evaluation counts to the wave's slot of the launch's count
 * (one atomic per wave). */
__device__ __forceinline__ void count_evals(unsigned long long *counter, unsigned long long n, uint32_t wid)
{
    for (int off = 32; off > 0; off >>= 1) n += __shfl_down(n, off);
    if (__lane_id() == 0 && n) atomicAdd(counter + wid % kEvalSlots * kEvalStride, n);
}

/* march.hip */
constexpr uint32_t kMaxPasses = 16;
constexpr size_t kPassRecBytes = 48;
struct MarchPlan {
    uint32_t n = 0;                   /* passes after the first; 0: the persistent levels */
    uint32_t subs = 0;                /* sub-lists per view */
    uint32_t K[kMaxPasses] = {};      /* lanes per ray of each pass, at least */
    uint32_t R[kMaxPasses] = {};      /* rounds of each pass (0: until the rays end) */
};
/* `rays`: of all views. */
MarchPlan march_plan(unsigned n_views, uint64_t rays);
/* Device memory of a launch's marching and parked rays. */
struct MarchBuffers {
    const void *view_table;
    void *cont;                       /* 2 x the views' cont_cap records */
    uint32_t *cont_counts;
    void *refine;
    uint32_t *refine_counts;
    uint32_t *counters;               /* evaluation counts */
};
int launch_march(lyap_ctx *ctx, const ViewDesc *views, unsigned n_views, const MarchPlan &mp,
                 const MarchBuffers &b, uint32_t W, int precision);
int launch_refine(lyap_ctx *ctx, unsigned n_views, uint32_t subs, uint64_t rays, const MarchBuffers &b,
                  uint32_t W, int precision, bool margin);

/* walk.hip */
int launch_walk(lyap_ctx *ctx, const void *view_table, unsigned n_views, uint64_t rays, uint32_t *counters,
                uint32_t W, int precision);

} /* namespace lyap */
