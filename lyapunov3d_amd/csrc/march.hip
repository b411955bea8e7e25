/*
 * march.hip - frames refined by bisection: march passes and refinement.
 *
 * A frame's rays march in passes, launches that advance every listed ray by
 * some rounds and list the rays still marching for the next pass; the rays
 * that found their opaque sample are parked and finished by one launch at the
 * end (refine_rays). In a round a ray has K lanes, which evaluate its next K
 * samples at once. The first pass takes the rays from the pixels, one lane
 * each, and one sample: half the rays that meet the box end there, so any
 * sample taken ahead would be wasted on them. The later passes choose K from
 * the number of rays listed, so that the chip's lanes are filled but no more
 * (a sample taken past a ray's end is wasted), and the last pass runs its
 * rays to their end. A ray's arithmetic is the same in every schedule, so
 * the bytes are too.
 */
#include <algorithm>
#include <cstdlib>

#include "render_common.hpp"

namespace lyap {
namespace {

/* A marching ray between passes (48 bytes, so that the two lists and the
 * parked rays' list take no more memory than the levels' lists). A ray refined
 * by bisection sits at C + V t with t = tb + m * dtb, and dtb is the step that
 * led there; its step is Fdt or Fdt / nearMultiplier by its near flag; every
 * sample so far was transparent and counted once, so the evaluations are the
 * index. What is left out is recomputed by the march's own expressions, bit
 * for bit. */
struct alignas(16) PassRec {
    uint32_t pix, flags_index;         /* near flag, kShortBit, march sample index [, m] */
    uint32_t m_or_Fdt;
    float Vx, Vy, Vz, t1, tb, dtb, a, c, l;
};
static_assert(sizeof(PassRec) == kPassRecBytes, "pass record size");

struct PassArgs {
    uint32_t n_views;
    uint32_t subs;                     /* sub-lists per view */
    uint32_t K;                        /* lanes per ray, at least */
    uint32_t rounds;                   /* rounds per ray (0: until the march ends) */
    uint32_t lanes;                    /* lanes a launch should fill */
    const PassRec *cont_in;            /* the rays to advance */
    const uint32_t *in_counts;         /* per view and sub-list, kHeadStride words apart */
    PassRec *cont_out;                 /* the rays still marching */
    uint32_t *out_counts;
    RefineRec *refine_out;
    uint32_t *refine_counts;           /* per view and sub-list, kHeadStride words apart */
    unsigned long long *eval_counter;
};

/* A ray's march state; every lane of its group holds the same copy. */
struct MarchRay {
    uint32_t pix, index, m;
    bool near_;
    F3 V;
    float t, t1, dt, Fdt, Ndt, last_step, a, c, l;
    /* samples lie at t = tb + m * dtb, rebased when the step length changes */
    float tb, dtb;
};

__device__ __forceinline__ float far_step(const ViewDesc &v, F3 V, float t0, float t1)
{
    return v.prm.stepMethod == 1 ? (t1 - t0) / v.prm.depth : sqrtf(mag2(V)) / v.prm.depth;
}

/* The march state of a ray that meets the box over [t0, t1]
 * (kernel.cu:281-314). */
__device__ __forceinline__ void begin_ray(const ViewDesc &v, uint32_t pix, F3 V, float t0, float t1, MarchRay &r)
{
    r.pix = pix;
    r.index = r.m = 0;
    r.near_ = false;
    r.V = V;
    r.t = r.tb = t0;
    r.t1 = t1;
    r.Fdt = far_step(v, V, t0, t1);
    r.dt = r.dtb = r.last_step = r.Fdt;
    r.Ndt = r.Fdt / v.prm.nearMultiplier;
    r.a = r.c = r.l = 0.f;
}

/* Up to kShort samples m (never above the index) and the index share a word,
 * which leaves one for the far step. Past them that step is computed from the
 * ray's length in the box again, whose six double divisions would cost the
 * passes of a short march 1 us each (frames of 512x512: 331 us against 320). */
constexpr uint32_t kShort = 0x8000u, kNearBit = 0x80000000u, kShortBit = 0x40000000u;

__device__ __forceinline__ void store_ray(const MarchRay &r, PassRec &q)
{
    const bool brief = r.index < kShort;
    q.pix = r.pix;
    q.flags_index = (brief ? kShortBit | r.index << 15 | r.m : r.index) | (r.near_ ? kNearBit : 0u);
    q.m_or_Fdt = brief ? __float_as_uint(r.Fdt) : r.m;
    q.Vx = r.V.x; q.Vy = r.V.y; q.Vz = r.V.z;
    q.t1 = r.t1; q.tb = r.tb; q.dtb = r.dtb;
    q.a = r.a; q.c = r.c; q.l = r.l;
}

__device__ __forceinline__ void load_ray(const ViewDesc &v, const PassRec &q, MarchRay &r)
{
    r.pix = q.pix;
    r.V = {q.Vx, q.Vy, q.Vz};
    r.near_ = (q.flags_index & kNearBit) != 0;
    r.t1 = q.t1;
    if (q.flags_index & kShortBit) {
        r.index = q.flags_index >> 15 & (kShort - 1u);
        r.m = q.flags_index & (kShort - 1u);
        r.Fdt = __uint_as_float(q.m_or_Fdt);
    } else {
        float t0 = 0.f, t1 = r.t1;
        if (v.prm.stepMethod == 1) (void)clip_box(f3(v.cam.C), r.V, v.prm.lMin, v.prm.lMax, t0, t1);
        r.index = q.flags_index & (kShortBit - 1u);
        r.m = q.m_or_Fdt;
        r.Fdt = far_step(v, r.V, t0, t1);
    }
    r.Ndt = r.Fdt / v.prm.nearMultiplier;
    r.dt = r.near_ ? r.Ndt : r.Fdt;
    r.tb = q.tb;
    r.dtb = r.last_step = q.dtb;
    r.t = r.tb + (float)r.m * r.dtb;
    r.a = q.a; r.c = q.c; r.l = q.l;
}

/* The next sample's t after a step of `step`; false when the step does not
 * change t (a grazing ray, or depth = inf), which would never leave the box. */
__device__ __forceinline__ bool advance(MarchRay &r, float step)
{
    if (step != r.dtb) {
        r.tb = r.t;
        r.dtb = step;
        r.m = 0;
    }
    const float tn = r.tb + (float)(r.m + 1u) * r.dtb;
    if (!(tn > r.t)) return false;
    r.t = tn;
    ++r.m;
    return true;
}

enum : int { R_NONE = 0, R_MARCH = 1, R_PARK = 2, R_MISS = 3 };

/* A wave's shares of the chaos and attractor sums. */
struct Shares {
    float c[64], a[64];
};

/* One round of the wave's rays: K samples each, then the state after the
 * samples the sequential method would have taken (kernel.cu:318-398).
 * `state` R_MARCH: the lane's ray is marching; on return R_MARCH, R_PARK (its
 * last sample is opaque: l_prev is the lambda before it) or R_MISS. `evals`:
 * the evaluations of a ray that ended. */
template <int W, int PREC>
__device__ __forceinline__ void march_round(const ViewDesc &v, MarchRay &r, int &state, float &l_prev,
                                            uint32_t &evals, uint32_t K, uint32_t rank, uint32_t gbase,
                                            Shares &sh)
{
    const LyapParams &prm = v.prm;
    const bool busy = state == R_MARCH;
    /* sample `rank`, taken ahead at the current step length; under jitter
     * the next step needs this sample's lambda */
    float ts = r.t;
    bool valid = busy;
    if (rank != 0) {
        const float tp = r.tb + (float)(r.m + rank - 1u) * r.dt;
        ts = r.tb + (float)(r.m + rank) * r.dt;
        valid = busy && prm.jitter == 0.0f && r.dt == r.dtb && ts > tp && !(ts > r.t1) &&
                r.index + rank < v.max_samples;
    }
    float lam = NAN;
    if (valid) {
        const F3 s = add(f3(v.cam.C), mul(r.V, ts));
        lam = eval_lambda<W, PREC>(v.e, s.x, s.y, s.z);
    }
    /* does the sample stop the run of transparent ones (opaque, invalid, a
     * near/far toggle, or jitter)? */
    const bool toggles = r.index + rank > 0u && r.Ndt != r.Fdt && (lam <= prm.nearThreshold) != r.near_;
    const bool ev = !valid || !(lam > prm.opaqueThreshold) || toggles || prm.jitter != 0.0f;
    const uint64_t kmask = K >= 64u ? ~0ull : ((1ull << K) - 1ull);
    const uint64_t evm = (__ballot(ev) >> gbase) & kmask;
    const uint32_t e = evm ? (uint32_t)__ffsll((unsigned long long)evm) - 1u : K;   /* transparent samples */
    const bool stopped = e < K;
    /* the sums: c += l above the chaos threshold, else a += l above the opaque
     * one (kernel.cu:370-375), over the samples taken, in order; a share that
     * adds to neither is +0, and adding +0 leaves a sum (never -0) unchanged */
    float sc = 0.0f, sa = 0.0f;
    if (valid && rank <= e && r.index + rank > 0u) {
        if (lam > prm.chaosThreshold) sc = lam;
        else if (lam > prm.opaqueThreshold) sa = lam;
    }
    float lam_e = lam, lam_p = lam;
    bool valid_e = valid;
    if (K == 1u) {
        r.c += sc;
        r.a += sa;
    } else {
        const bool any_c = __ballot(sc != 0.0f) != 0, any_a = __ballot(sa != 0.0f) != 0;
        wave_sync_lds();                           /* the last round's shares have been read */
        sh.c[gbase + rank] = sc;
        sh.a[gbase + rank] = sa;
        wave_sync_lds();
        const uint32_t n = busy ? (stopped ? e + 1u : K) : 0u;
        if (K >= 4u) {
            for (uint32_t j = 0; __ballot(j < n) != 0; j += 4u) {
                /* j < K: a group's four shares lie in its own slots */
                if (any_c) {
                    const float4 q = *reinterpret_cast<const float4 *>(&sh.c[gbase + j]);
                    r.c += q.x; r.c += q.y; r.c += q.z; r.c += q.w;
                }
                if (any_a) {
                    const float4 q = *reinterpret_cast<const float4 *>(&sh.a[gbase + j]);
                    r.a += q.x; r.a += q.y; r.a += q.z; r.a += q.w;
                }
            }
        } else {
            r.c += sh.c[gbase]; r.c += sh.c[gbase + 1u];
            r.a += sh.a[gbase]; r.a += sh.a[gbase + 1u];
        }
        lam_e = __shfl(lam, (int)(gbase + (stopped ? e : K - 1u)));
        lam_p = __shfl(lam, (int)(gbase + (e ? e - 1u : 0u)));
        valid_e = ((__ballot(valid) >> (gbase + (stopped ? e : 0u))) & 1ull) != 0;
    }
    if (!busy) return;
    l_prev = e ? lam_p : r.l;
    if (e) r.last_step = r.dt;
    r.index += e;
    const uint32_t ahead = stopped ? e : K - 1u;
    if (ahead) {
        r.m += ahead;
        r.t = r.tb + (float)r.m * r.dt;
    }
    evals = r.index;
    if (!stopped) {
        /* all transparent: on to the sample after them */
        r.l = lam_p;
        if (r.index >= v.max_samples || !advance(r, r.dt) || r.t > r.t1) state = R_MISS;
        return;
    }
    if (!valid_e) {
        /* the step to sample e left the box or could not advance */
        state = R_MISS;
        return;
    }
    evals = r.index + 1u;
    r.l = lam_e;
    if (r.index > 0u) {
        if (lam_e <= prm.nearThreshold && !r.near_) { r.near_ = true; r.dt = r.Ndt; }
        else if (lam_e > prm.nearThreshold && r.near_) { r.near_ = false; r.dt = r.Fdt; }
    }
    if (!(lam_e > prm.opaqueThreshold)) {
        state = R_PARK;
        return;
    }
    float step = r.dt;
    if (prm.jitter != 0.0f) {
        float jit = lam_e - truncf(lam_e);
        if (jit < 0) jit = (float)(1.0 - (double)(jit * prm.jitter));
        else jit = (float)(1.0 + (double)(jit * prm.jitter));
        if (__builtin_isfinite(jit)) step = r.dt * jit;
    }
    if (!advance(r, step)) {
        state = R_MISS;
        return;
    }
    r.last_step = step;
    ++r.index;
    if (r.t > r.t1 || r.index >= v.max_samples) state = R_MISS;
}

/* Lists the rays still marching (`cont`) and parks those that found their
 * opaque sample (`park`; both for one lane per ray) on view vi's sub-lists:
 * the one of this block's index, which waves of one XCD share, then the next
 * ones while a sub-list is full. A view's sub-lists hold all its rays
 * together, and a full one has every entry written, so each ray finds a
 * place. One atomic per wave, list and try. */
__device__ __forceinline__ void append_rays(const ViewDesc &v, uint32_t vi, const MarchRay &r, float l_prev,
                                            uint32_t evals, bool cont, bool park, const PassArgs &a)
{
    const uint32_t lane = __lane_id();
    const uint64_t below = (1ull << lane) - 1ull;
    const uint32_t cont_sub = v.cont_cap / a.subs;
    for (uint32_t tries = 0; tries < a.subs; ++tries) {
        const uint64_t cm = __ballot(cont), pm = __ballot(park);
        if ((cm | pm) == 0) return;
        const uint32_t sub = (blockIdx.x + tries) % a.subs;
        const uint32_t slot0 = (vi * a.subs + sub) * kHeadStride;
        uint32_t base = 0;
        if (lane == 0 && cm) base = atomicAdd(a.out_counts + slot0, (uint32_t)__popcll(cm));
        if (lane == 1 && pm) base = atomicAdd(a.refine_counts + slot0, (uint32_t)__popcll(pm));
        const uint32_t cb = uniform((uint32_t)__shfl((int)base, 0)), pb = uniform((uint32_t)__shfl((int)base, 1));
        if (cont) {
            const uint32_t slot = cb + (uint32_t)__popcll(cm & below);
            if (slot < cont_sub) {
                PassRec q;
                store_ray(r, q);
                a.cont_out[(size_t)v.cont_base + sub * cont_sub + slot] = q;
                cont = false;
            }
        }
        if (park) {
            const uint32_t slot = pb + (uint32_t)__popcll(pm & below);
            if (slot < v.refine_cap) {
                RefineRec q;
                q.pix = r.pix;
                q.evals = evals;
                q.Vx = r.V.x;
                q.Vy = r.V.y;
                q.Vz = r.V.z;
                q.lo = r.t - r.last_step;
                q.hi = r.t;
                q.l_hi = r.l;
                q.dt = r.dt;
                q.a = r.a;
                q.c = r.c;
                q.l_lo = l_prev;
                a.refine_out[(size_t)v.refine_base + sub * v.refine_cap + slot] = q;
                park = false;
            }
        }
    }
}

/* The first pass: every pixel ray of every view, one lane each and one sample
 * (views start at multiples of 256 in this grid). Rays that miss the box are
 * written at once. */
template <int W, int PREC>
__global__ __launch_bounds__(64) void march_start(const ViewDesc *__restrict__ views, PassArgs a)
{
    const uint32_t lane = __lane_id();
    const uint32_t first = blockIdx.x * 64u;
    /* the view: ray_base rises with the view index and view 0 begins at 0 */
    uint32_t vi = 0;
    if (a.n_views <= 64u) {
        const bool before = lane < a.n_views && views[lane].ray_base <= first;
        vi = uniform((uint32_t)__popcll(__ballot(before)) - 1u);
    } else {
        while (vi + 1u < a.n_views && views[uniform(vi + 1u)].ray_base <= first) ++vi;
        vi = uniform(vi);
    }
    const ViewDesc &v = views[vi];
    const uint32_t id = first - v.ray_base + lane;
    uint32_t pix = 0;
    F3 V = {0.f, 0.f, 0.f};
    float t0 = 0.f, t1 = 0.f;
    const int kind = id < v.n_rays ? ray_setup(v, id, pix, V, t0, t1) : (int)RAY_PAD;
    if (kind == RAY_MISS) write_miss(v, pix, 0u);
    if (__ballot(kind == RAY_HIT) == 0) return;
    MarchRay r;
    begin_ray(v, pix, V, t0, t1, r);
    int state = kind == RAY_HIT ? R_MARCH : R_NONE;
    float l_prev = 0.f;
    uint32_t evals = 0;
    __shared__ Shares sh;              /* not used at one lane per ray */
    march_round<W, PREC>(v, r, state, l_prev, evals, 1u, 0u, lane, sh);
    if (state == R_MISS) write_miss(v, pix, evals);
    append_rays(v, vi, r, l_prev, evals, state == R_MARCH, state == R_PARK, a);
    count_evals(a.eval_counter, state == R_MISS ? evals : 0u, blockIdx.x);
}

/* `rounds` rounds (0: until the march ends) for every listed ray. Vector
 * instructions bound it, and six waves per SIMD run them best: five (90
 * registers) take 857 us for a frame of 1024x1024 and 326 for 512x512, six 830
 * and 325, eight, with registers spilled, 831 and 337. */
template <int W, int PREC>
__global__ __launch_bounds__(256, W == 16 && PREC == LYAP_PREC_PRODUCT ? 6 : 1)
void march_pass(const ViewDesc *__restrict__ views, PassArgs a)
{
    __shared__ Shares shares[4];
    Shares &sh = shares[threadIdx.x >> 6];
    const uint32_t lane = __lane_id();
    const uint32_t n_waves = gridDim.x * 4u;
    const uint32_t wid = uniform(blockIdx.x * 4u + threadIdx.x / 64u);
    /* up to 64 lists, held across the wave: lane j has list j's count */
    const uint32_t pairs = a.n_views * a.subs;
    uint32_t n = 0;
    if (lane < pairs) n = min(a.in_counts[lane * kHeadStride], views[lane / a.subs].cont_cap / a.subs);
    uint32_t total = n;
    for (int off = 32; off > 0; off >>= 1) total += (uint32_t)__shfl_xor((int)total, off);
    total = uniform(total);
    if (total == 0) return;
    /* more lanes per ray while the launch's lanes have room for them */
    uint32_t K = a.K;
    while (K < 64u && (uint64_t)total * (2u * K) <= a.lanes) K *= 2u;
    K = uniform(K);
    const uint32_t per = 64u / K;                 /* rays per wave and round */
    const uint32_t rank = lane % K;
    const uint32_t gbase = lane - rank;
    const ChunkMap cm = chunk_map(n, per, lane);
    unsigned long long done = 0;
    for (uint32_t c = wid; c < cm.total; c += n_waves) {
        uint32_t acc, p, cnt;
        chunk_find(cm, c, per, p, acc, cnt);
        const uint32_t vi = uniform(p / a.subs);
        const ViewDesc &v = views[vi];
        const uint32_t i = (c - acc) * per + lane / K;
        int state = i < cnt ? R_MARCH : R_NONE;
        MarchRay r{};
        if (state == R_MARCH)
            load_ray(v, a.cont_in[(size_t)v.cont_base + (p % a.subs) * (v.cont_cap / a.subs) + i], r);
        float l_prev = 0.f;
        uint32_t evals = 0;
        bool missed = false, parked = false;
        for (uint32_t round = 0;;) {
            march_round<W, PREC>(v, r, state, l_prev, evals, K, rank, gbase, sh);
            if (state == R_MISS) missed = true;
            if (state == R_PARK) parked = true;
            if (state != R_MARCH) state = R_NONE;
            ++round;
            if (round == a.rounds || __ballot(state == R_MARCH) == 0) break;
        }
        if (missed && rank == 0) {
            write_miss(v, r.pix, evals);
            done += evals;
        }
        append_rays(v, vi, r, l_prev, evals, state == R_MARCH && rank == 0, parked && rank == 0, a);
    }
    count_evals(a.eval_counter, done, wid);
}

/* ---- refinement launch -------------------------------------------------- */

struct RefineArgs {
    uint32_t n_views;
    uint32_t subs;                     /* sub-lists per view */
    const RefineRec *recs;
    const uint32_t *counts;            /* per view and sub-list, kHeadStride words apart */
    unsigned long long *eval_counter;
};

/* Records of view-sub-region pair p that the march launches wrote. */
__device__ __forceinline__ uint32_t refine_count(const ViewDesc *__restrict__ views,
                                                 const RefineArgs &a, uint32_t p)
{
    return uniform(min(a.counts[p * kHeadStride], views[uniform(p / a.subs)].refine_cap));
}

template <int W, int PREC, bool MARGIN>
__device__ __forceinline__ float refine_eval(const ViewDesc &v, F3 sp, float thr)
{
    float lam = eval_lambda<W, PREC>(v.e, sp.x, sp.y, sp.z);
    if (MARGIN && PREC != LYAP_PREC_FP64 && !(__builtin_fabsf(lam - thr) >= v.margin))
        lam = eval_fp64_call<W>(v.e, sp.x, sp.y, sp.z);
    return lam;
}

/* Finishes the parked rays, G lanes per ray and 64 / G rays of one view per
 * wave: the bisection of [lo, hi] (the midpoint rule), the six normal
 * samples in the order x-, x+, y-, y+, z-, z+ (kernel.cu:456-473), the hit
 * record and its colour. With two lanes the first evaluates the midpoint of
 * a bisection trip and the second the midpoint of the half the crossing of
 * the line through lambda at lo and hi falls in; when that half is the one
 * the first sample chooses, the trip resolves two levels. The normal then
 * takes three trips, the minus samples on the first lane and the plus samples
 * on the second. The arithmetic is the march kernel's, step for step, so the
 * bytes are those of refining in place. Vector instructions bound it (a record
 * is read once per 14 samples), so registers are held to eight waves per SIMD:
 * 64 frames of 512x512 44.0 ms against 46.6 with seven. Two lanes halve a small launch's
 * chain of evaluations; one lane evaluates nothing it does not need (14
 * samples a ray instead of about 17), which a launch that fills the chip many
 * times over is bound by. */
template <int W, int PREC, bool MARGIN, int G>
__global__ __launch_bounds__(256, W == 16 && PREC == LYAP_PREC_PRODUCT && !MARGIN ? 8 : 1)
void refine_rays(const ViewDesc *__restrict__ views, RefineArgs a)
{
    constexpr uint32_t per = 64u / G;
    const uint32_t lane = __lane_id();
    const uint32_t side = lane % G;            /* 0: midpoints, minus normal samples */
    const uint32_t n_waves = gridDim.x * 4u;
    const uint32_t wid = uniform(blockIdx.x * 4u + threadIdx.x / 64u);
    const uint32_t pairs = a.n_views * a.subs;
    const bool held = pairs <= 64u;
    ChunkMap cm{0u, 0u, 0u};
    uint32_t total = 0;
    if (held) {
        uint32_t n = 0;
        if (lane < pairs) n = min(a.counts[lane * kHeadStride], views[lane / a.subs].refine_cap);
        cm = chunk_map(n, per, lane);
        total = cm.total;
    } else {
        for (uint32_t p = 0; p < pairs; ++p) total += (refine_count(views, a, p) + per - 1u) / per;
    }
    unsigned long long done = 0;
    for (uint32_t t = wid; t < total; t += n_waves) {
        uint32_t acc = 0, p = 0, n = 0;
        if (held) {
            chunk_find(cm, t, per, p, acc, n);
        } else {
            for (; p < pairs; ++p) {
                n = refine_count(views, a, p);
                const uint32_t nt = (n + per - 1u) / per;
                if (t < acc + nt) break;
                acc += nt;
            }
        }
        const ViewDesc &v = views[uniform(p / a.subs)];
        const uint32_t i = (t - acc) * per + lane / G;
        const bool has = i < n;
        RefineRec q{};
        if (has) q = a.recs[(size_t)v.refine_base + (p % a.subs) * v.refine_cap + i];
        const F3 C = f3(v.cam.C);
        const F3 V = {q.Vx, q.Vy, q.Vz};
        const float thr = v.prm.opaqueThreshold;
        float lo = q.lo, hi = q.hi, l_hi = q.l_hi, l_lo = q.l_lo;
        uint32_t evals = q.evals;
        /* a ray's lanes hold the same interval; trips are wave-uniform */
        for (int k = 0; __ballot(has && k < v.bisect_steps) != 0;) {
            const bool go = has && k < v.bisect_steps;
            const float mid = lo + (hi - lo) * 0.5f;
            float at = mid;
            bool guess_lo = false;
            if (G == 2) {
                /* the half the line's crossing falls in, and its midpoint */
                const float f = (l_lo - thr) / (l_lo - l_hi);
                guess_lo = !(lo + (hi - lo) * f > mid);
                const float mid2 = guess_lo ? lo + (mid - lo) * 0.5f : mid + (hi - mid) * 0.5f;
                if (side) at = mid2;
            }
            float lam = 0.f;
            if (go) lam = refine_eval<W, PREC, MARGIN>(v, add(C, mul(V, at)), thr);
            const float lm = G == 2 ? __shfl(lam, (int)(lane & ~1u)) : lam;
            const float lg = G == 2 ? __shfl(lam, (int)(lane | 1u)) : 0.f;
            if (go) {
                ++evals;
                ++k;
                const bool opaque = !(lm > thr);
                if (opaque) { hi = mid; l_hi = lm; }
                else { lo = mid; l_lo = lm; }
                if (G == 2 && k < v.bisect_steps && opaque == guess_lo) {
                    /* the guessed half is the one taken: its midpoint, formed
                     * from the same interval, is the next level's */
                    ++evals;
                    ++k;
                    const float m2 = lo + (hi - lo) * 0.5f;
                    if (!(lg > thr)) { hi = m2; l_hi = lg; }
                    else { lo = m2; l_lo = lg; }
                }
            }
        }
        const F3 P = add(C, mul(V, hi));
        const float h = (v.normal_h > 0.0f) ? v.normal_h : q.dt * v.prm.gradient;
        F3 g = {0.f, 0.f, 0.f};
        for (uint32_t k = 0; k < 6u / G; ++k) {
            const uint32_t axis = G == 2 ? k : k >> 1;
            const bool plus = G == 2 ? side != 0 : (k & 1u) != 0;
            const float off = plus ? h : -h;
            F3 sp = P;
            if (axis == 0) sp.x = P.x + off;
            else if (axis == 1) sp.y = P.y + off;
            else sp.z = P.z + off;
            float lam = 0.f;
            if (has) lam = eval_lambda<W, PREC>(v.e, sp.x, sp.y, sp.z);
            float d;
            if (G == 2) {
                const float lminus = __shfl(lam, (int)(lane & ~1u));
                const float lplus = __shfl(lam, (int)(lane | 1u));
                d = -lminus;
                d = d + lplus;
            } else {
                const float before = axis == 0 ? g.x : (axis == 1 ? g.y : g.z);
                d = plus ? before + lam : -lam;
            }
            if (axis == 0) g.x = d;
            else if (axis == 1) g.y = d;
            else g.z = d;
        }
        if (has && side == 0) {
            const F3 N = normalized(g);
            write_hit(v, q.pix, evals + 6u, P, N, hi, l_hi, q.a, q.c);
            const C4 cc = shade(P, N, q.a, q.c, v.cam, v.lights, v.num_lights);
            LyapRGBA px;
            px.r = to_u8(cc.x);
            px.g = to_u8(cc.y);
            px.b = to_u8(cc.z);
            px.a = to_u8(cc.w);
            v.rgba[q.pix] = px;
            done += evals + 6u;
        }
    }
    count_evals(a.eval_counter, done, wid);
}

/* Pass sequences, "lanes per ray x rounds" and 0 rounds for the last one.
 * Below kManyRays a launch's time is its chain of passes and refinement trips:
 * it takes few passes, samples ahead, and two refining lanes per ray. Below
 * kSmallRays, where a pass raises its lanes per ray far above the minimum, its
 * first passes take one or two rounds, as most rays end within those samples;
 * above it, where they do not, four rounds save listing the rays again. Short
 * / long first passes, in us per frame: 74x370 plain 270 / 300, 170x278 plain
 * 309 / 342, 256x256 product 251 / 256, plain 380 / 408, FP64 377 / 414,
 * 512x512 307 / 293, 768x768 544 / 530, 1024x1024 853 / 793.
 * From kManyRays on the chip is full whatever the lanes, and a sample taken
 * past a ray's end costs what a needed one does: one lane per ray for as long
 * as enough rays march, in passes short enough that the lanes of ended rays do
 * not idle long, and one refining lane. Long first passes / one lane: 256x256
 * 265 / 335, 512x512 320 / 371, 1024x1024 796 / 864, 1448x1448 1499 / 1464,
 * 2048x2048 2900 / 2584; 64 frames of 512x512 48700 / 38600. The march kernel
 * in levels takes 355, 509 and 1765 us for the first three and 51900 for the
 * 64. */
constexpr uint64_t kSmallRays = 200000;
constexpr uint64_t kManyRays = 1800000;
/* Blocks: a pass of many rays gets kManyTurns grids' worth, and the refinement
 * several per slot, so that a slot whose blocks had cheap rays takes another
 * one: 64 frames of 512x512 take 41.4 ms with one grid each and 37.3 so. */
constexpr uint32_t kManyTurns = 4, kFewRefine = 16, kManyRefine = 64;
const char *const kSmallPasses = "2x1,2x2,4x2,8x2,16x4,32x4,64x0";
const char *const kFewPasses = "2x4,4x4,8x4,16x4,32x4,64x4,64x0";
const char *const kManyPasses = "1x4,1x4,1x8,1x8,1x16,1x16,2x16,2x16,4x16,8x16,16x8,64x0";

} /* namespace */

/* The passes after march_start. LYAP_MARCH_PASSES overrides their sequence
 * for experiments: comma-separated "K" or "KxR" (at least K lanes per ray; R
 * rounds, 0: until the rays end; one without it); "0" switches the passes
 * off. The last pass always runs its rays to the end. */
MarchPlan march_plan(unsigned n_views, uint64_t rays)
{
    MarchPlan mp;
    if (n_views > 64u) return mp;      /* a wave holds the counts of 64 lists */
    mp.subs = n_views <= 8u ? 8u : 64u / n_views;
    static const char *env = std::getenv("LYAP_MARCH_PASSES");
    const char *c = env ? env : rays < kSmallRays ? kSmallPasses : rays < kManyRays ? kFewPasses : kManyPasses;
    if (c[0] == '0' && c[1] == 0) return mp;
    while (*c && mp.n < kMaxPasses) {
        char *e = nullptr;
        const unsigned long k = std::strtoul(c, &e, 10);
        if (k == 0 || k > 64 || (k & (k - 1))) return MarchPlan{};
        unsigned long r = 1;
        if (*e == 'x') r = std::strtoul(e + 1, &e, 10);
        mp.K[mp.n] = (uint32_t)k;
        mp.R[mp.n] = (uint32_t)r;
        ++mp.n;
        if (*e != ',') break;
        c = e + 1;
    }
    if (mp.n) mp.R[mp.n - 1] = 0;
    return mp;
}

template <int W, int PREC>
static uint32_t pass_blocks_per_cu()
{
    static int cached = -1;
    if (cached < 0) {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &n, reinterpret_cast<const void *>(&march_pass<W, PREC>), 256, 0) != hipSuccess ||
            n <= 0)
            n = 2;
        cached = n;
    }
    return (uint32_t)cached;
}

/* Enqueues march_start and the passes: march_start lists the rays still
 * marching under counts[0], pass p reads those listed under counts[p] and
 * lists what is left under counts[p + 1] (the two buffers alternate). */
int launch_march(lyap_ctx *ctx, const ViewDesc *views, unsigned n_views, const MarchPlan &mp,
                 const MarchBuffers &b, uint32_t W, int precision)
{
    uint64_t cap_total = 0, rays = 0, all = 0;
    for (unsigned i = 0; i < n_views; ++i) {
        cap_total += views[i].cont_cap;
        all += views[i].n_rays;
        rays += (views[i].n_rays + 255u) / 256u * 256u;
    }
    PassRec *buf[2] = {(PassRec *)b.cont, (PassRec *)b.cont + cap_total};
    const uint32_t pass_words = n_views * mp.subs * kHeadStride;
    const uint32_t cus = ctx->num_cus > 0 ? (uint32_t)ctx->num_cus : 256u;
    const uint32_t turns = all >= kManyRays ? kManyTurns : 1u;
    PassArgs a{};
    a.n_views = n_views;
    a.subs = mp.subs;
    a.refine_out = (RefineRec *)b.refine;
    a.refine_counts = b.refine_counts;
    a.eval_counter = (unsigned long long *)b.counters;
    a.cont_out = buf[0];
    a.out_counts = b.cont_counts;
    const ViewDesc *table = (const ViewDesc *)b.view_table;
    int rc = timing_mark(ctx);
    if (rc) return rc;
#define LYAP_LAUNCH(WW, PP)                                                                            \
    hipLaunchKernelGGL((march_start<WW, PP>), dim3((uint32_t)((rays + 63u) / 64u)), dim3(64), 0,        \
                       ctx->stream, table, a)
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
    rc = timing_mark(ctx);
    if (rc) return rc;
    for (uint32_t p = 0; p < mp.n; ++p) {
        a.K = mp.K[p];
        a.rounds = mp.R[p];
        a.cont_in = buf[p & 1u];
        a.in_counts = b.cont_counts + p * pass_words;
        a.cont_out = buf[(p + 1u) & 1u];
        a.out_counts = b.cont_counts + (p + 1u) * pass_words;
        rc = timing_mark(ctx);
        if (rc) return rc;
#define LYAP_LAUNCH(WW, PP)                                                                            \
    do {                                                                                               \
        const uint32_t blocks = cus * pass_blocks_per_cu<WW, PP>();                                    \
        a.lanes = blocks * 256u;                                                                       \
        hipLaunchKernelGGL((march_pass<WW, PP>), dim3(blocks * turns), dim3(256), 0, ctx->stream, table, a); \
    } while (0)
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
        rc = timing_mark(ctx);
        if (rc) return rc;
    }
    return LYAP_OK;
}

/* The refinement launch over the parked rays, `subs` sub-lists per view. */
int launch_refine(lyap_ctx *ctx, unsigned n_views, uint32_t subs, uint64_t rays, const MarchBuffers &b,
                  uint32_t W, int precision, bool margin)
{
    const bool many = rays >= kManyRays;
    RefineArgs ra{};
    ra.n_views = n_views;
    ra.subs = subs;
    ra.recs = (const RefineRec *)b.refine;
    ra.counts = b.refine_counts;
    ra.eval_counter = (unsigned long long *)b.counters;
    const uint32_t cus = ctx->num_cus > 0 ? (uint32_t)ctx->num_cus : 256u;
    const uint32_t blocks = cus * (many ? kManyRefine : kFewRefine);
#define LYAP_LAUNCH(WW, PP, MM)                                                                     \
    do {                                                                                            \
        if (many)                                                                                   \
            hipLaunchKernelGGL((refine_rays<WW, PP, MM, 1>), dim3(blocks), dim3(256), 0, ctx->stream, \
                               (const ViewDesc *)b.view_table, ra);                                 \
        else                                                                                        \
            hipLaunchKernelGGL((refine_rays<WW, PP, MM, 2>), dim3(blocks), dim3(256), 0, ctx->stream, \
                               (const ViewDesc *)b.view_table, ra);                                 \
    } while (0)
    if (W == 16) {
        if (precision == LYAP_PREC_PLAIN) LYAP_LAUNCH(16, LYAP_PREC_PLAIN, false);
        else if (precision == LYAP_PREC_PRODUCT && margin) LYAP_LAUNCH(16, LYAP_PREC_PRODUCT, true);
        else if (precision == LYAP_PREC_PRODUCT) LYAP_LAUNCH(16, LYAP_PREC_PRODUCT, false);
        else LYAP_LAUNCH(16, LYAP_PREC_FP64, false);
    } else {
        if (precision == LYAP_PREC_PLAIN) LYAP_LAUNCH(32, LYAP_PREC_PLAIN, false);
        else if (precision == LYAP_PREC_PRODUCT && margin) LYAP_LAUNCH(32, LYAP_PREC_PRODUCT, true);
        else if (precision == LYAP_PREC_PRODUCT) LYAP_LAUNCH(32, LYAP_PREC_PRODUCT, false);
        else LYAP_LAUNCH(32, LYAP_PREC_FP64, false);
    }
#undef LYAP_LAUNCH
    LYAP_HIP(ctx, hipGetLastError());
    return LYAP_OK;
}

} /* namespace lyap */
