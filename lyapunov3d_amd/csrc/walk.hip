/*
 * walk.hip - frames refined by the reference's reversing walk, one lane per
 * ray.
 *
 * The reference's method (kernel.cu:156-486 with the walk of :402-441 and
 * the step jitter of :334-352): the next march step depends on the last
 * sample's lambda, so a ray's samples cannot be taken ahead and lanes beyond
 * one per ray have nothing to do.
 */
#include "render_common.hpp"

namespace lyap {
namespace {

enum : int { W_IDLE = 0, W_MARCH = 1, W_WALK = 2, W_NORMAL = 3 };

constexpr uint32_t kMaxWalk = 64;

/* A ray's state, in the order it needs it: the march, then the walk's
 * interval and step, then the normal's sums. */
struct WalkRay {
    int phase;
    uint32_t evals, index, k;
    bool near_, sign;
    F3 V, P;
    float t, t1, dt, Fdt, Ndt, a, c, l;
    float Qdt, Qt0, Qt1, minQdt;
    F3 QdV;
    float h;
    F3 g;
};

__device__ __forceinline__ void begin_normal(const ViewDesc &v, WalkRay &r)
{
    r.phase = W_NORMAL;
    r.k = 0;
    r.h = (v.normal_h > 0.0f) ? v.normal_h : r.dt * v.prm.gradient;
}

/* walk loop test (kernel.cu:420) */
__device__ __forceinline__ bool keeps_walking(const WalkRay &r)
{
    return r.k < kMaxWalk && r.t <= r.Qt1 && r.t >= r.Qt0 && (r.Qdt <= -r.minQdt || r.Qdt >= r.minQdt);
}

/* Takes the march sample l at (t, P): the sums, the near step, then the next
 * position, or the walk when l is opaque. Returns false when the ray left the
 * box (or could not advance). */
__device__ __forceinline__ bool take_march(const ViewDesc &v, WalkRay &r, float l)
{
    const LyapParams &prm = v.prm;
    ++r.evals;
    r.l = l;
    if (r.index > 0) {
        /* kernel.cu:370-384 */
        if (l > prm.chaosThreshold) r.c += l;
        else if (l > prm.opaqueThreshold) r.a += l;
        if (l <= prm.nearThreshold && !r.near_) { r.near_ = true; r.dt = r.Ndt; }
        else if (l > prm.nearThreshold && r.near_) { r.near_ = false; r.dt = r.Fdt; }
    }
    if (l > prm.opaqueThreshold) {
        float step = r.dt;
        if (prm.jitter != 0.0f) {
            float jit = l - truncf(l);
            if (jit < 0) jit = (float)(1.0 - (double)(jit * prm.jitter));
            else jit = (float)(1.0 + (double)(jit * prm.jitter));
            if (__builtin_isfinite(jit)) step = r.dt * jit;
        }
        if (!(r.t + step > r.t)) return false;
        r.t += step;
        r.P = add(r.P, mul(r.V, step));
        ++r.index;
        return !(r.t > r.t1 || r.index >= v.max_samples);
    }
    r.phase = W_WALK;
    r.k = 0;
    r.sign = false;
    r.Qdt = r.dt * -0.5f;
    r.QdV = mul(r.V, r.Qdt);
    r.Qt1 = r.t;
    r.Qt0 = r.t - r.dt;
    r.minQdt = r.dt / prm.refine;
    if (!keeps_walking(r)) begin_normal(v, r);
    return true;
}

/* Takes the walk's sample l at (t + Qdt, P + QdV) (kernel.cu:420-441). */
__device__ __forceinline__ void take_walk(const ViewDesc &v, WalkRay &r, float l)
{
    const float thr = v.prm.opaqueThreshold;
    r.t += r.Qdt;
    r.P = add(r.P, r.QdV);
    ++r.evals;
    ++r.k;
    r.l = l;
    if (l == thr) {
        begin_normal(v, r);
        return;
    }
    const bool s = !(l < thr);
    if (s != r.sign) {
        r.Qdt *= -0.5f;
        r.QdV = mul(r.QdV, -0.5f);
    }
    r.sign = s;
    if (!keeps_walking(r)) begin_normal(v, r);
}

/* Takes normal sample k, in the order x-, x+, y-, y+, z-, z+
 * (kernel.cu:456-473). */
__device__ __forceinline__ void take_normal(WalkRay &r, float l)
{
    const uint32_t n = r.k;
    const float sl = (n & 1u) ? l : -l;
    if (n < 2) r.g.x = (n == 0) ? sl : r.g.x + sl;
    else if (n < 4) r.g.y = (n == 2) ? sl : r.g.y + sl;
    else r.g.z = (n == 4) ? sl : r.g.z + sl;
    ++r.k;
    ++r.evals;
    if (r.k >= 6u) r.phase = W_IDLE;
}

/* One wave per 8x8 pixel block, one lane per ray from its first sample to
 * its last; each trip of the loop evaluates one lambda per lane whose ray has
 * not ended, whichever phase the ray is in. The ray's record and colour are
 * written once the wave's rays have all ended, with all lanes.
 *
 * Bound by the longest ray's chain of samples on a small frame (1,000 waves
 * of a 320 x 200 frame, one per SIMD, 207 samples at most), so the trip holds
 * nothing but the evaluation and the state's update: no sample goes through
 * LDS, no tile is claimed, no ray is handed over: 0.68 ms at 18 + 120
 * iterations per sample. The persistent levels, which give such a frame 16
 * lanes per ray, 15 of them idle, took 9.2 ms. */
template <int W, int PREC>
__global__ __launch_bounds__(64) void walk_rays(const ViewDesc *__restrict__ views, uint32_t n_views,
                                                unsigned long long *eval_counter)
{
    const uint32_t lane = __lane_id();
    const uint32_t first = blockIdx.x * 64u;
    uint32_t vi = 0;
    while (vi + 1u < n_views && views[uniform(vi + 1u)].ray_base <= first) ++vi;
    const ViewDesc &v = views[uniform(vi)];
    const uint32_t id = first - v.ray_base + lane;
    uint32_t pix = 0;
    WalkRay r;
    float t0 = 0.f;
    r.t1 = 0.f;
    const int kind = id < v.n_rays ? ray_setup(v, id, pix, r.V, t0, r.t1) : (int)RAY_PAD;
    if (kind == RAY_MISS) write_miss(v, pix, 0u);
    /* kernel.cu:281-314 */
    r.phase = kind == RAY_HIT ? W_MARCH : W_IDLE;
    r.evals = r.index = r.k = 0;
    r.near_ = r.sign = false;
    r.t = t0;
    r.P = add(f3(v.cam.C), mul(r.V, t0));
    r.a = r.c = r.l = 0.f;
    r.Fdt = v.prm.stepMethod == 1 ? (r.t1 - t0) / v.prm.depth : sqrtf(mag2(r.V)) / v.prm.depth;
    r.dt = r.Fdt;
    r.Ndt = r.dt / v.prm.nearMultiplier;
    bool missed = false;
    while (__ballot(r.phase != W_IDLE) != 0) {
        F3 sp = r.P;
        if (r.phase == W_WALK) {
            sp = add(r.P, r.QdV);
        } else if (r.phase == W_NORMAL) {
            const float off = (r.k & 1u) ? r.h : -r.h;
            if (r.k < 2u) sp.x = r.P.x + off;
            else if (r.k < 4u) sp.y = r.P.y + off;
            else sp.z = r.P.z + off;
        }
        if (r.phase != W_IDLE) {
            const float lam = eval_lambda<W, PREC>(v.e, sp.x, sp.y, sp.z);
            if (r.phase == W_MARCH) {
                if (!take_march(v, r, lam)) {
                    r.phase = W_IDLE;
                    missed = true;
                }
            } else if (r.phase == W_WALK) {
                take_walk(v, r, lam);
            } else {
                take_normal(r, lam);
            }
        }
    }
    if (missed) {
        write_miss(v, pix, r.evals);
    } else if (kind == RAY_HIT) {
        const F3 N = normalized(r.g);
        write_hit(v, pix, r.evals, r.P, N, r.t, r.l, r.a, r.c);
        const C4 cc = shade(r.P, N, r.a, r.c, v.cam, v.lights, v.num_lights);
        LyapRGBA px;
        px.r = to_u8(cc.x);
        px.g = to_u8(cc.y);
        px.b = to_u8(cc.z);
        px.a = to_u8(cc.w);
        v.rgba[pix] = px;
    }
    count_evals(eval_counter, kind == RAY_HIT ? r.evals : 0u, blockIdx.x);
}

} /* namespace */

/* `rays`: the views' rays, each view from a multiple of 256 on (ray_base). */
int launch_walk(lyap_ctx *ctx, const void *view_table, unsigned n_views, uint64_t rays, uint32_t *counters,
                uint32_t W, int precision)
{
#define LYAP_LAUNCH(WW, PP)                                                                          \
    hipLaunchKernelGGL((walk_rays<WW, PP>), dim3((uint32_t)((rays + 63u) / 64u)), dim3(64), 0,        \
                       ctx->stream, (const ViewDesc *)view_table, n_views, (unsigned long long *)counters)
    if (W == 16) {
        if (precision == LYAP_PREC_PLAIN) LYAP_LAUNCH(16, LYAP_PREC_PLAIN);
        else if (precision == LYAP_PREC_PRODUCT) LYAP_LAUNCH(16, LYAP_PREC_PRODUCT);
        else LYAP_LAUNCH(16, LYAP_PREC_FP64);
    } else {
        if (precision == LYAP_PREC_PLAIN) LYAP_LAUNCH(32, LYAP_PREC_PLAIN);
        else if (precision == LYAP_PREC_PRODUCT) LYAP_LAUNCH(32, LYAP_PREC_PRODUCT);
        else LYAP_LAUNCH(32, LYAP_PREC_FP64);
    }
#undef LYAP_LAUNCH
    LYAP_HIP(ctx, hipGetLastError());
    return LYAP_OK;
}

} /* namespace lyap */
