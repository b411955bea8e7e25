/*
 * lyap_device.hpp - the per-point Lyapunov exponent on gfx950.
 *
 * One lane evaluates one point. The reference routine is lyap4d
 * (kernel.cu:108-154): x0 = 0.5, `settle` steps of x <- r x (1 - x), then
 * `accum` steps summing ln|r_n (1 - 2 x_{n+1})| (the derivative uses the new
 * iterate, kernel.cu:143-144); |x - 0.5| < 1e-8 after the settle returns 0
 * (kernel.cu:138); a non-finite sum returns NaN (kernel.cu:147-149); the
 * sequence position wraps at the -1 terminator and carries over from the
 * settle into the accumulation (kernel.cu:133-134, 141-142).
 *
 * Three arithmetic forms:
 *
 *  plain<L>    FP32 iterate, one hardware log2 per accumulated step. The
 *              reference method in FP32; the baseline kernel.
 *
 *  product<L>  FP32 iterate in u = 1 - 2x, where the map becomes
 *              u' = (1 - r/2) + (r/2) u^2 and the derivative factor is
 *              r_n u_{n+1}. |u| <= 1 while 0 <= r <= 4, so the running product
 *              M of |u| only shrinks between renormalisations: it is carried
 *              as an FP32 mantissa plus an int32 exponent, renormalised every
 *              block of whole periods (up to 40 steps for the volumes, one
 *              16- or 32-slot window for the render), and a block that ends
 *              below the smallest normal float (where gradual underflow could
 *              have cost bits) is recomputed with a renormalisation per step.
 *              Renormalising is exact, so the block length changes no bit. The ln|r_n| terms depend only on the
 *              letter, so they are added once per letter with host-computed
 *              counts. One log2 per evaluation instead of one per step.
 *              Per accumulated step: one multiply (u^2), one FMA, one
 *              multiply into M.
 *
 *  fp64<L>     FP64 map with exactly the reference's operation order
 *              ((r*v)*(1-v), no fused multiply-add; the whole library is
 *              built with -ffp-contract=off), so the orbit is bitwise the one
 *              an IEEE double CPU computes. The derivative r(1 - 2v) only
 *              feeds the log sum and is formed with one fma; the log sum is
 *              carried as a product with exponent renormalisation every 8
 *              steps, which changes lambda only by rounding (~1e-15).
 *
 * Sequence handling: the period L is a template parameter, so the
 * coefficients of each sequence position sit in VGPRs and the step loop is
 * unrolled over one period. The letters themselves are wave-uniform (kernel
 * arguments in SGPRs); a position's coefficient is picked from the lane's
 * (x, y, z, d) once per evaluation.
 */
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "lyap.h"
#include "sequence.hpp"

namespace lyap {

constexpr float kLn2f = 0.693147180559945309f;
constexpr double kLn2 = 0.693147180559945309417232121458;
/* A product block ending below the smallest normal float may have lost bits
 * to gradual underflow; one ending at or above it did not, since |u| <= 1
 * keeps the product non-increasing within the block. Such a block is
 * recomputed with a renormalisation per step. */
constexpr float kUnderflowGuard = 0x1p-126f;

/* The per-period kernels keep the running product scaled by 2^120 within a
 * block of steps: |u| <= 1 only shrinks it, so a block has 2^246 of range
 * before gradual underflow could cost bits, and scaling by a power of two is
 * exact. (Started at [0.5, 1), 30-step blocks in stable regions fell below
 * 2^-126 about half the time.) */
constexpr float kProductScale = 0x1p120f;
constexpr int kProductScaleExp = 120;

/* Whether a block's product has to be redone: it ended below the smallest
 * normal float, where bits may be lost, or at infinity or NaN (the orbit of a
 * point with r > 4, in a volume reaching past 4, can escape [0, 1], and then
 * |u| > 1 grows fast and may overflow between renormalisations where its
 * factors are finite). Redone per step the product stays finite while its
 * factors are, so block lengths never change a bit, and lambda is finite
 * exactly when every factor is (as with the reference's sum of logs). One
 * compare: the class is not "positive normal". The window forms of the
 * persistent launch keep a compare with the guard: their samples lie in the
 * [lMin, lMax] box (at most an ulp past it). */
__device__ __forceinline__ bool bad_block(float M)
{
    return !__builtin_amdgcn_classf(M, 0x100);
}

/* Wave-uniform description of one lambda evaluation: iteration counts,
 * sequence, and host-derived loop bounds. Built by make_eval_desc(). */
struct EvalDesc {
    uint32_t settle, accum;
    float d;
    int32_t L;
    int32_t letters[LYAP_MAX_SEQ];
    /* settle = settle_periods * L + settle_rem */
    uint32_t settle_periods, settle_rem;
    /* accumulation: positions [head_begin, head_end) of the period the settle
     * ended in, then acc_periods full periods, then positions [0, tail). */
    uint32_t head_begin, head_end;
    uint32_t acc_periods, tail;
    /* first part of the window for the convergence check: the head plus
     * half_periods full periods (half_steps steps) */
    uint32_t half_periods, half_steps;
    /* 1 / accum and 1 / steps of the window's two parts, rounded to nearest */
    double inv_accum, inv_half1, inv_half2;
    /* occurrences of letters A..D in the whole window and in its first part */
    float count[4];
    float count_half[4];
    /* Blocked layout for the period-agnostic kernels: a block is B steps, a
     * whole number of periods that fits the kernel's coefficient window W;
     * position j of a block uses letter wletters[j] = letters[j mod L].
     * settle = set_blocks * B + set_rem; the accumulation finishes that block
     * (positions [head_lo, head_hi)), runs acc_blocks blocks, then positions
     * [0, acc_rem). */
    int32_t wletters[LYAP_MAX_SEQ];
    /* the same as bit masks: bit j of wmask[k] is set when wletters[j] == k,
     * so a kernel builds its coefficients from one 16-byte scalar load */
    uint32_t wmask[4];
    uint32_t W, B;
    uint32_t set_blocks, set_rem;
    uint32_t head_lo, head_hi;
    uint32_t acc_blocks, acc_rem;
};

inline void rebuild_blocks(EvalDesc *e, uint32_t W);

/* Host: derive the loop bounds. Returns false for an unusable sequence. */
inline bool make_eval_desc(EvalDesc *e, const LyapParams &prm, const int32_t *seq)
{
    const int L = sequence_period(seq);
    if (L == 0) return false;
    *e = EvalDesc{};
    e->settle = prm.settle;
    e->accum = prm.accum;
    e->d = prm.d;
    e->L = L;
    for (int j = 0; j < L; ++j) e->letters[j] = seq[j];
    e->settle_periods = prm.settle / L;
    e->settle_rem = prm.settle % L;
    uint32_t left = prm.accum;
    e->head_begin = e->settle_rem;
    e->head_end = e->settle_rem;
    if (e->settle_rem != 0) {
        const uint32_t h = (uint32_t)L - e->settle_rem;
        const uint32_t take = left < h ? left : h;
        e->head_end = e->settle_rem + take;
        left -= take;
    }
    e->acc_periods = left / L;
    e->tail = left % L;
    e->half_periods = e->acc_periods / 2;
    e->half_steps = (e->head_end - e->head_begin) + e->half_periods * (uint32_t)L;
    e->inv_accum = 1.0 / (double)prm.accum;
    e->inv_half1 = 1.0 / (double)e->half_steps;
    e->inv_half2 = 1.0 / (double)(prm.accum - e->half_steps);
    /* letter counts */
    for (int k = 0; k < 4; ++k) { e->count[k] = 0.f; e->count_half[k] = 0.f; }
    for (uint32_t j = e->head_begin; j < e->head_end; ++j) {
        e->count[seq[j]] += 1.f;
        e->count_half[seq[j]] += 1.f;
    }
    for (int j = 0; j < L; ++j) {
        e->count[seq[j]] += (float)e->acc_periods;
        e->count_half[seq[j]] += (float)e->half_periods;
    }
    for (uint32_t j = 0; j < e->tail; ++j) e->count[seq[j]] += 1.f;
    rebuild_blocks(e, L <= 16 ? 16u : 32u);
    return true;
}

/* Host: blocked layout for a coefficient window of W (16 or 32) positions. */
inline void rebuild_blocks(EvalDesc *e, uint32_t W)
{
    const uint32_t L = (uint32_t)e->L;
    e->W = W;
    /* a 32-slot window with a period of at most 16 takes two 16-slot blocks
     * at a time, so the FP64 form, renormalised at half and end of each
     * block, renormalises after the same steps in either window */
    e->B = (W > 16 && L <= 16) ? 2u * (L * (16u / L)) : L * (W / L);
    for (uint32_t k = 0; k < 4; ++k) e->wmask[k] = 0;
    for (uint32_t j = 0; j < (uint32_t)LYAP_MAX_SEQ; ++j) {
        e->wletters[j] = e->letters[j % L];
        e->wmask[e->wletters[j] & 3] |= 1u << j;
    }
    e->set_blocks = e->settle / e->B;
    e->set_rem = e->settle % e->B;
    uint32_t left = e->accum;
    e->head_lo = e->head_hi = 0;
    if (e->set_rem != 0) {
        const uint32_t h = e->B - e->set_rem;
        const uint32_t take = left < h ? left : h;
        e->head_lo = e->set_rem;
        e->head_hi = e->set_rem + take;
        left -= take;
    }
    e->acc_blocks = left / e->B;
    e->acc_rem = left % e->B;
}

/* Lane's value of the letter at position j, from the letter masks (uniform;
 * one scalar load for all positions): a bit-field insert per letter, its mask
 * the position's bit spread over a scalar register. */
__device__ __forceinline__ void load_masks(uint32_t (&m)[4], const EvalDesc &e)
{
#pragma unroll
    for (int k = 0; k < 4; ++k) m[k] = e.wmask[k];
}
__device__ __forceinline__ uint32_t spread_bit(uint32_t m, int j)
{
    return (uint32_t)((int32_t)(m << (31 - j)) >> 31);
}
__device__ __forceinline__ float pick_mask(const uint32_t (&m)[4], int j, float x, float y, float z, float d)
{
    const uint32_t ma = spread_bit(m[0], j), mb = spread_bit(m[1], j), mc = spread_bit(m[2], j);
    uint32_t v = (__float_as_uint(z) & mc) | (__float_as_uint(d) & ~mc);
    v = (__float_as_uint(y) & mb) | (v & ~mb);
    v = (__float_as_uint(x) & ma) | (v & ~ma);
    return __uint_as_float(v);
}

/* ---- blocks of periods and settled orbits -------------------------------
 *
 * The per-period kernels run blocks of block_periods<L>() whole periods, a
 * power of two of them. The map is a function of the iterate alone at a given
 * sequence position, so an iterate that comes back bit for bit to where it was
 * a block earlier repeats that block for ever: in the stable regions the
 * rounded orbit reaches its attractor exactly after about 24 ln 2 / |lambda|
 * steps (53 in double), and an attractor of 1, 2, 4, ... periods divides the
 * block. Once that is so in every lane of a wave the wave skips the rest of
 * the settle, and in the accumulation applies the block's factors (product
 * form), logs (plain) or derivatives (double), kept from one run of the
 * block, without iterating the map: the same operations on the accumulator in
 * the same order, so the same bits, in one instruction a step instead of three
 * (product) or five (plain, double). Of the 256^3 volume over [2.5, 4]^3 47 % of the voxels and 35 % of
 * the 4x4x4 bricks have settled by step 256, 61 % and 44 % by the end. */
template <int L>
constexpr int block_periods()
{
    int h = 1;
    while (2 * h * L <= 40) h *= 2;
    return h;
}

/* Whether every lane's iterate came back to where the block started. */
template <typename T>
__device__ __forceinline__ bool settled(T now, T before)
{
    return __ballot(now != before) == 0;
}

/* ---- plain FP32: one log2 per accumulated step ------------------------- */

template <int L>
__device__ __forceinline__ float lambda_plain(float x, float y, float z,
                                              const EvalDesc &e)
{
    float r[L], m2r[L];
    uint32_t m[4];
    load_masks(m, e);
#pragma unroll
    for (int j = 0; j < L; ++j) {
        r[j] = pick_mask(m, j, x, y, z, e.d);
        m2r[j] = -2.0f * r[j];
    }
    float v = 0.5f;
    for (uint32_t p = 0; p < e.settle_periods; ++p) {
#pragma unroll
        for (int j = 0; j < L; ++j) v = r[j] * __builtin_fmaf(-v, v, v);
    }
#pragma unroll
    for (int j = 0; j < L; ++j)
        if ((uint32_t)j < e.settle_rem) v = r[j] * __builtin_fmaf(-v, v, v);

    if (v == 0.5f) return 0.0f / (float)e.accum;   /* kernel.cu:138 in FP32 */

    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < L; ++j) {
        if ((uint32_t)j >= e.head_begin && (uint32_t)j < e.head_end) {
            v = r[j] * __builtin_fmaf(-v, v, v);
            s += __builtin_amdgcn_logf(__builtin_fabsf(__builtin_fmaf(m2r[j], v, r[j])));
        }
    }
    /* A loop of one period: in straight lines of a block the logs of several
     * waves meet in the quarter-rate unit (10.0 ns a step with eight waves
     * per SIMD against 8.9). It runs in stretches, to an eighth, a quarter,
     * half and all of the window, so that looking for a settled orbit between
     * them costs the others nothing. */
    constexpr uint32_t H = block_periods<L>();
    uint32_t done = 0;
    const auto run_to = [&](uint32_t end) {
        for (; done < end; ++done) {
#pragma unroll
            for (int j = 0; j < L; ++j) {
                v = r[j] * __builtin_fmaf(-v, v, v);
                s += __builtin_amdgcn_logf(__builtin_fabsf(__builtin_fmaf(m2r[j], v, r[j])));
            }
        }
    };
    for (uint32_t part = 8; part > 1; part >>= 1) {
        const uint32_t end = e.acc_periods / part;
        if (end < done + H || e.acc_periods - end < 2 * H) continue;
        run_to(end - H);
        const float v0 = v;
        run_to(end);
        if (settled(v, v0)) {
            float lg[H * L];
#pragma unroll
            for (int i = 0; i < (int)H * L; ++i) {
                v = r[i % L] * __builtin_fmaf(-v, v, v);
                lg[i] = __builtin_amdgcn_logf(__builtin_fabsf(__builtin_fmaf(m2r[i % L], v, r[i % L])));
            }
            for (; done + H <= e.acc_periods; done += H) {
#pragma unroll
                for (int i = 0; i < (int)H * L; ++i) s += lg[i];
            }
            break;
        }
    }
    run_to(e.acc_periods);
#pragma unroll
    for (int j = 0; j < L; ++j) {
        if ((uint32_t)j < e.tail) {
            v = r[j] * __builtin_fmaf(-v, v, v);
            s += __builtin_amdgcn_logf(__builtin_fabsf(__builtin_fmaf(m2r[j], v, r[j])));
        }
    }
    const float lam = s * kLn2f / (float)e.accum;
    return __builtin_isfinite(lam) ? lam : __builtin_nanf("");
}

/* ---- FP32 u-form with a mantissa/exponent product ---------------------- */

struct ProductState {
    float M;     /* mantissa of the running product of |u| */
    int E;       /* its binary exponent */
};

__device__ __forceinline__ void renorm(ProductState &st)
{
    st.E += __builtin_amdgcn_frexp_expf(st.M);
    st.M = __builtin_amdgcn_frexp_mantf(st.M);
}

/* a / n for a whole number n < 2^32, given y = 1 / n rounded to nearest, in 3
 * operations instead of the division's dozen. The estimate a * y is within
 * 1.5 ulp, its residual a - n q fits a double and so is exact, and the
 * corrected quotient is off by less than 2^-52 ulp before it is rounded,
 * while a / n lies at least 2^-34 ulp from any rounding boundary: the result
 * is the correctly rounded quotient. n = 0 and a non-finite a give NaN. */
__device__ __forceinline__ double divide_by(double a, double n, double y)
{
    const double q = a * y;
    return __builtin_fma(__builtin_fma(-n, q, a), y, q);
}

/* ln of the product plus the letter terms, divided by n (inv = 1 / n); NaN if
 * not finite. */
__device__ __forceinline__ float finish_product(const ProductState &st,
                                                const float lg[4],
                                                const float cnt[4], uint32_t n, double inv)
{
    double t = (double)st.E + (double)__builtin_amdgcn_logf(st.M);
#pragma unroll
    for (int k = 0; k < 4; ++k)
        if (cnt[k] != 0.0f) t += (double)cnt[k] * (double)lg[k];
    const float lam = (float)divide_by(t * kLn2, (double)n, inv);
    return __builtin_isfinite(lam) ? lam : __builtin_nanf("");
}

/* Result of a product-form evaluation. half1/half2 are the lambdas of the
 * two parts of the window (NaN when a part is empty). */
struct ProductResult {
    float lam;
    float half1, half2;
};

/* FP32 maps in u = 1 - 2x with b = r/2. The volume form u' = b u^2 + a with
 * a = 1 - b (a multiply and an FMA) is what every volume evaluator uses (the
 * per-period kernels and the window form of volume blocks in the persistent
 * launch), so they give the same bits for the same voxel; the render's form
 * u' = 1 + b (u^2 - 1) (two FMAs) needs no a and so half the coefficient
 * registers. Renormalising the product is exact, so block lengths change no
 * bit; only the map's rounding does. */
__device__ __forceinline__ float vmap(float u, float a, float b)
{
    return __builtin_fmaf(b, u * u, a);
}

__device__ __forceinline__ float umap(float u, float b)
{
    return __builtin_fmaf(b, __builtin_fmaf(u, u, -1.0f), 1.0f);
}

/* The end of a block that started at st.M * kProductScale and ended at Mb. */
__device__ __forceinline__ void renorm_scaled(ProductState &st, float Mb)
{
    st.E += __builtin_amdgcn_frexp_expf(Mb) - kProductScaleExp;
    st.M = __builtin_amdgcn_frexp_mantf(Mb);
}

/* `n` full periods of the product in blocks of about 12 steps, a lane's bad
 * block recomputed with a renormalisation per step. */
template <int L>
__device__ __forceinline__ void product_periods_slow(float &u, ProductState &st, const float (&a)[L],
                                                     const float (&b)[L], uint32_t n)
{
    constexpr uint32_t S = L < 12 ? (12 + L / 2) / L : 1;
    for (uint32_t left = n; left;) {
        const uint32_t cnt = left < S ? left : S;
        left -= cnt;
        const float u0 = u;
        float M = st.M * kProductScale;
        for (uint32_t k = 0; k < cnt; ++k) {
#pragma unroll
            for (int j = 0; j < L; ++j) {
                u = vmap(u, a[j], b[j]);
                M *= __builtin_fabsf(u);
            }
        }
        if (!bad_block(M)) {
            renorm_scaled(st, M);
        } else {
            float w = u0;
            for (uint32_t k = 0; k < cnt; ++k) {
#pragma unroll
                for (int j = 0; j < L; ++j) {
                    w = vmap(w, a[j], b[j]);
                    st.M *= __builtin_fabsf(w);
                    renorm(st);
                }
            }
        }
    }
}

/* `n` full periods of the product. Straight-line blocks with one branch each
 * (a taken branch costs a wave about 20 clocks of instruction fetch, as much
 * as five steps: 11.2, 7.8 and 6.0 ns a step in lines of 5, 8 and 30 steps
 * with one wave per SIMD, 4.7, 4.4 and 3.6 ns with eight), until a lane has a
 * bad block, the wave has settled, or less than a block is left. */
template <int L>
__device__ __forceinline__ void product_periods(float &u, ProductState &st, const float (&a)[L],
                                                const float (&b)[L], uint32_t n)
{
    constexpr uint32_t H = block_periods<L>();
    uint32_t left = n;
    if (left >= H) {
        float w[H * L];                /* the block's iterates */
        float u0;
        ProductState s0;
        bool bad, cycle;
        do {
            u0 = u;
            s0 = st;
            float M = st.M * kProductScale;
#pragma unroll
            for (int i = 0; i < (int)H * L; ++i) {
                w[i] = vmap(i ? w[i - 1] : u, a[i % L], b[i % L]);
                M *= __builtin_fabsf(w[i]);
            }
            u = w[H * L - 1];
            bad = __ballot(bad_block(M)) != 0;
            cycle = settled(u, u0);
            renorm_scaled(st, M);
            left -= H;
        } while (!bad & !cycle & (left >= H));
        if (bad) {
            /* back to the state before the block */
            u = u0;
            st = s0;
            left += H;
        } else if (cycle) {
            while (left >= H) {
                s0 = st;
                float M = st.M * kProductScale;
#pragma unroll
                for (int i = 0; i < (int)H * L; ++i) M *= __builtin_fabsf(w[i]);
                if (__ballot(bad_block(M)) != 0) break;
                renorm_scaled(st, M);
                left -= H;
            }
        }
    }
    product_periods_slow<L>(u, st, a, b, left);
}

/* `n` full settle periods, in the same straight-line blocks. */
template <int L>
__device__ __forceinline__ void settle_periods(float &u, const float (&a)[L], const float (&b)[L],
                                               uint32_t n)
{
    constexpr uint32_t H = block_periods<L>();
    uint32_t left = n;
    if (left >= H) {
        bool cycle;
        do {
            const float u0 = u;
#pragma unroll
            for (int i = 0; i < (int)H * L; ++i) u = vmap(u, a[i % L], b[i % L]);
            cycle = settled(u, u0);
            left -= H;
        } while (!cycle & (left >= H));
        if (cycle) left %= H;
    }
    for (; left; --left) {
#pragma unroll
        for (int j = 0; j < L; ++j) u = vmap(u, a[j], b[j]);
    }
}

template <int L, bool HALVES>
__device__ __forceinline__ ProductResult lambda_product(float x, float y,
                                                        float z,
                                                        const EvalDesc &e)
{
    float a[L], b[L];
    uint32_t m[4];
    load_masks(m, e);
#pragma unroll
    for (int j = 0; j < L; ++j) {
        b[j] = 0.5f * pick_mask(m, j, x, y, z, e.d);
        a[j] = 1.0f - b[j];
    }
    float u = 0.0f;
    settle_periods<L>(u, a, b, e.settle_periods);
#pragma unroll
    for (int j = 0; j < L; ++j)
        if ((uint32_t)j < e.settle_rem) u = vmap(u, a[j], b[j]);

    ProductResult res;
    /* kernel.cu:138: |x - 0.5| < 1e-8 is |u| < 2e-8 */
    if (__builtin_fabsf(u) < 2e-8f) {
        res.lam = 0.0f / (float)e.accum;
        res.half1 = res.half2 = res.lam;
        return res;
    }

    ProductState st{1.0f, 0};
    /* head: the rest of the period the settle ended in, renormalised per step */
#pragma unroll
    for (int j = 0; j < L; ++j) {
        if ((uint32_t)j >= e.head_begin && (uint32_t)j < e.head_end) {
            u = vmap(u, a[j], b[j]);
            st.M *= __builtin_fabsf(u);
            renorm(st);
        }
    }
    ProductState st_half{1.0f, 0};
    if (HALVES) {
        product_periods<L>(u, st, a, b, e.half_periods);
        st_half = st;
        product_periods<L>(u, st, a, b, e.acc_periods - e.half_periods);
    } else {
        product_periods<L>(u, st, a, b, e.acc_periods);
    }
#pragma unroll
    for (int j = 0; j < L; ++j) {
        if ((uint32_t)j < e.tail) {
            u = vmap(u, a[j], b[j]);
            st.M *= __builtin_fabsf(u);
            renorm(st);
        }
    }

    float lg[4];
    lg[0] = __builtin_amdgcn_logf(__builtin_fabsf(x));
    lg[1] = __builtin_amdgcn_logf(__builtin_fabsf(y));
    lg[2] = __builtin_amdgcn_logf(__builtin_fabsf(z));
    lg[3] = __builtin_amdgcn_logf(__builtin_fabsf(e.d));
    res.lam = finish_product(st, lg, e.count, e.accum, e.inv_accum);
    res.half1 = res.half2 = res.lam;
    if (HALVES) {
        const uint32_t n1 = e.half_steps, n2 = e.accum - e.half_steps;
        float c2[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) c2[k] = e.count[k] - e.count_half[k];
        ProductState second;
        second.E = st.E - st_half.E;
        second.M = st.M / st_half.M;
        res.half1 = n1 ? finish_product(st_half, lg, e.count_half, n1, e.inv_half1) : __builtin_nanf("");
        res.half2 = n2 ? finish_product(second, lg, c2, n2, e.inv_half2) : __builtin_nanf("");
    }
    return res;
}

/* ---- FP64 with the reference's operation order ------------------------- */

struct ProductState64 {
    double M;
    int E;
};

__device__ __forceinline__ void renorm64(ProductState64 &st)
{
    st.E += __builtin_amdgcn_frexp_exp(st.M);
    st.M = __builtin_amdgcn_frexp_mant(st.M);
}

/* Periods of an FP64 block: a power of two of them making up to 20 steps (40
 * registers of derivatives), at least one. */
template <int L>
constexpr int block_periods64()
{
    int h = 1;
    while (2 * h * L <= 20) h *= 2;
    return h;
}

/* CYCLES: look for settled orbits. The FP64 pass over a list leaves that out:
 * its points were listed because they have not settled (and the derivatives
 * kept cost it a wave per SIMD: 2.34 ms against 2.30 for 6.1 M points). */
template <int L, bool CYCLES>
__device__ __forceinline__ double lambda_fp64(float xf, float yf, float zf,
                                              const EvalDesc &e)
{
    double r[L], m2r[L];
    uint32_t m[4];
    load_masks(m, e);
#pragma unroll
    for (int j = 0; j < L; ++j) {
        r[j] = (double)pick_mask(m, j, xf, yf, zf, e.d);
        m2r[j] = -2.0 * r[j];        /* exact */
    }
    double v = 0.5;
    for (uint32_t p = 0; p < e.settle_periods; ++p) {
#pragma unroll
        for (int j = 0; j < L; ++j) v = (r[j] * v) * (1.0 - v);
    }
#pragma unroll
    for (int j = 0; j < L; ++j)
        if ((uint32_t)j < e.settle_rem) v = (r[j] * v) * (1.0 - v);

    const double off = v - 0.5;
    if (!(off <= -1e-8 || off >= 1e-8)) return 0.0 / (double)e.accum;

    ProductState64 st{1.0, 0};
#pragma unroll
    for (int j = 0; j < L; ++j) {
        if ((uint32_t)j >= e.head_begin && (uint32_t)j < e.head_end) {
            v = (r[j] * v) * (1.0 - v);
            st.M *= __builtin_fabs(__builtin_fma(m2r[j], v, r[j]));
            renorm64(st);
        }
    }
    /* factors are at most max|r| * max|1 - 2v|; 8 of them cannot leave the
     * double range for coordinates of float magnitude (or the orbit escapes,
     * which makes lambda NaN either way) */
    constexpr uint32_t H = block_periods64<L>();
    uint32_t done = 0;
    const auto run_to = [&](uint32_t end) {
        for (; done < end; ++done) {
#pragma unroll
            for (int j = 0; j < L; ++j) {
                v = (r[j] * v) * (1.0 - v);
                st.M *= __builtin_fabs(__builtin_fma(m2r[j], v, r[j]));
                if (((j + 1) & 7) == 0) renorm64(st);
            }
            if ((L & 7) != 0) renorm64(st);
        }
    };
    for (uint32_t part = 8; CYCLES && part > 1; part >>= 1) {
        const uint32_t end = e.acc_periods / part;
        if (end < done + H || e.acc_periods - end < 2 * H) continue;
        run_to(end - H);
        const double v0 = v;
        run_to(end);
        if (settled(v, v0)) {
            double f[H * L];
#pragma unroll
            for (int i = 0; i < (int)H * L; ++i) {
                v = (r[i % L] * v) * (1.0 - v);
                f[i] = __builtin_fabs(__builtin_fma(m2r[i % L], v, r[i % L]));
            }
            for (; done + H <= e.acc_periods; done += H) {
#pragma unroll
                for (int i = 0; i < (int)H * L; ++i) {
                    st.M *= f[i];
                    if (((i % L + 1) & 7) == 0 || (i + 1) % L == 0) renorm64(st);
                }
            }
            break;
        }
    }
    run_to(e.acc_periods);
#pragma unroll
    for (int j = 0; j < L; ++j) {
        if ((uint32_t)j < e.tail) {
            v = (r[j] * v) * (1.0 - v);
            st.M *= __builtin_fabs(__builtin_fma(m2r[j], v, r[j]));
            renorm64(st);
        }
    }
    const double lam = ((double)st.E * kLn2 + log(st.M)) / (double)e.accum;
    return __builtin_isfinite(lam) ? lam : __builtin_nan("");
}

/* ======================================================================== */
/* Period-agnostic forms: one compiled loop for every period L <= W.         */
/* ======================================================================== */

/* Steps of a block at positions [lo, hi) (FULL: [0, B), where every block
 * has at least W/2 + 1 steps, so only the upper half is guarded). */
template <int W, bool FULL>
__device__ __forceinline__ bool in_block(int j, uint32_t lo, uint32_t hi)
{
    if (FULL) return j <= W / 2 || (uint32_t)j < hi;
    return (uint32_t)j >= lo && (uint32_t)j < hi;
}

/* The coefficients of a window of W slots, b_j = r_j / 2. */
template <int W>
__device__ __forceinline__ void load_half_r(float (&b)[W], float x, float y, float z, const EvalDesc &e)
{
    const float hx = 0.5f * x, hy = 0.5f * y, hz = 0.5f * z, hd = 0.5f * e.d;
    uint32_t m[4];
    load_masks(m, e);
#pragma unroll
    for (int j = 0; j < W; ++j) b[j] = pick_mask(m, j, hx, hy, hz, hd);
}

/* Calls f.template go<N>() for n in [LO, HI], found by halving (n is
 * wave-uniform, so each test is a scalar branch). */
template <int LO, int HI, class F>
__device__ __forceinline__ void with_value(uint32_t n, F &f)
{
    if constexpr (LO == HI) {
        f.template go<LO>();
    } else {
        constexpr int MID = (LO + HI) / 2;
        if (n <= (uint32_t)MID) with_value<LO, MID>(n, f);
        else with_value<MID + 1, HI>(n, f);
    }
}

/* Calls f.template go<B>() with B the block length Bv, one of (W/2, W]. A
 * full block then runs exactly B unguarded steps. */
template <int W, class F>
__device__ __forceinline__ void with_block_len(uint32_t Bv, F &f)
{
    with_value<W / 2 + 1, W>(Bv, f);
}

/* Calls f.template go<N>() for n in [1, W); nothing for n = 0. Partial
 * blocks are specialised by their start or length this way, so none of
 * their steps carries a per-step guard. */
template <int W, class F>
__device__ __forceinline__ void with_len(uint32_t n, F &f)
{
    if (n != 0) with_value<1, W - 1>(n, f);
}

/* n full settle blocks of B steps. The loops of the window forms are one
 * block long: a launch of the march starts with a cold instruction cache, and
 * with runs of two blocks (and the redo apart from them) a 256 x 256 frame's
 * passes took 28 % longer, fetching code they run a few times. */
template <int W>
struct SettleFull {
    float &u;
    const float (&c)[W];
    uint32_t n;
    template <int B>
    __device__ __forceinline__ void go()
    {
        for (uint32_t k = 0; k < n; ++k) {
#pragma unroll
            for (int j = 0; j < B; ++j) u = umap(u, c[j]);
        }
    }
};

/* Window positions [LO, HI) of the product form; positions past W/2 are
 * guarded by j < hi when GUARD (they may lie past a block of B < W). A lane
 * whose block ends below the smallest normal float redoes it with a
 * renormalisation per step. */
template <int W, int LO, int HI, bool GUARD>
__device__ __forceinline__ void product_range(float &u, ProductState &st, const float (&c)[W], uint32_t hi)
{
    const float u0 = u;
    const ProductState s0 = st;
#pragma unroll
    for (int j = LO; j < HI; ++j) {
        if (!GUARD || j <= W / 2 || (uint32_t)j < hi) {
            u = umap(u, c[j]);
            st.M *= __builtin_fabsf(u);
        }
    }
    if (st.M < kUnderflowGuard) {
        /* |u| <= 1 keeps M monotone within the block, so ending above the
         * guard means no step went below it */
        float w = u0;
        st = s0;
#pragma unroll
        for (int j = LO; j < HI; ++j) {
            if (!GUARD || j <= W / 2 || (uint32_t)j < hi) {
                w = umap(w, c[j]);
                st.M *= __builtin_fabsf(w);
                renorm(st);
            }
        }
    }
    renorm(st);
}

/* The window positions [lo, hi), any 0 <= lo <= hi <= W. */
template <int W>
__device__ __forceinline__ void product_block(float &u, ProductState &st, const float (&c)[W],
                                              uint32_t lo, uint32_t hi)
{
    const float u0 = u;
    const ProductState s0 = st;
#pragma unroll
    for (int j = 0; j < W; ++j) {
        if ((uint32_t)j >= lo && (uint32_t)j < hi) {
            u = umap(u, c[j]);
            st.M *= __builtin_fabsf(u);
        }
    }
    if (st.M < kUnderflowGuard) {
        float w = u0;
        st = s0;
#pragma unroll
        for (int j = 0; j < W; ++j) {
            if ((uint32_t)j >= lo && (uint32_t)j < hi) {
                w = umap(w, c[j]);
                st.M *= __builtin_fabsf(w);
                renorm(st);
            }
        }
    }
    renorm(st);
}

/* n full product blocks of B steps. */
template <int W>
struct ProductFull {
    float &u;
    ProductState &st;
    const float (&c)[W];
    uint32_t n;
    template <int B>
    __device__ __forceinline__ void go()
    {
        for (uint32_t k = 0; k < n; ++k) product_range<W, 0, B, false>(u, st, c, 0);
    }
};

/* Settle steps [0, N) / product steps [0, N) / the rest of a block from N. */
template <int W>
struct SettlePrefix {
    float &u;
    const float (&c)[W];
    template <int N>
    __device__ __forceinline__ void go()
    {
#pragma unroll
        for (int j = 0; j < N; ++j) u = umap(u, c[j]);
    }
};

template <int W>
struct ProductPrefix {
    float &u;
    ProductState &st;
    const float (&c)[W];
    template <int N>
    __device__ __forceinline__ void go() { product_range<W, 0, N, false>(u, st, c, 0); }
};

template <int W>
struct ProductHead {
    float &u;
    ProductState &st;
    const float (&c)[W];
    uint32_t hi;
    template <int N>
    __device__ __forceinline__ void go() { product_range<W, N, W, true>(u, st, c, hi); }
};

/* FP32 product form, any period L <= W, with the render's map. */
template <int W>
__device__ __forceinline__ float lambda_product_w(float x, float y, float z,
                                                  const EvalDesc &e)
{
    float c[W];
    load_half_r<W>(c, x, y, z, e);
    float u = 0.0f;
    {
        SettleFull<W> f{u, c, e.set_blocks};
        with_block_len<W>(e.B, f);
    }
    {
        SettlePrefix<W> f{u, c};
        with_len<W>(e.set_rem, f);
    }
    if (__builtin_fabsf(u) < 2e-8f) return 0.0f / (float)e.accum;   /* kernel.cu:138 */
    ProductState st{1.0f, 0};
    if (e.head_hi == e.B) {
        /* the usual head: the rest of the block the settle ended in */
        ProductHead<W> f{u, st, c, e.B};
        with_len<W>(e.head_lo, f);
    } else {
        product_block<W>(u, st, c, e.head_lo, e.head_hi);
    }
    {
        ProductFull<W> f{u, st, c, e.acc_blocks};
        with_block_len<W>(e.B, f);
    }
    {
        ProductPrefix<W> f{u, st, c};
        with_len<W>(e.acc_rem, f);
    }
    float lg[4];
    lg[0] = __builtin_amdgcn_logf(__builtin_fabsf(x));
    lg[1] = __builtin_amdgcn_logf(__builtin_fabsf(y));
    lg[2] = __builtin_amdgcn_logf(__builtin_fabsf(z));
    lg[3] = __builtin_amdgcn_logf(__builtin_fabsf(e.d));
    return finish_product(st, lg, e.count, e.accum, e.inv_accum);
}

/* FP32 x-form with one log2 per accumulated step (the reference method). */
template <int W, bool FULL>
__device__ __forceinline__ void plain_block(float &v, float &s, const float (&r)[W],
                                            uint32_t lo, uint32_t hi, bool acc)
{
#pragma unroll
    for (int j = 0; j < W; ++j) {
        if (in_block<W, FULL>(j, lo, hi)) {
            v = r[j] * __builtin_fmaf(-v, v, v);
            if (acc) s += __builtin_amdgcn_logf(__builtin_fabsf(__builtin_fmaf(-2.0f * r[j], v, r[j])));
        }
    }
}

/* n full blocks of B steps of the x-form, accumulating when ACC. */
template <int W, bool ACC>
struct PlainFull {
    float &v;
    float &s;
    const float (&r)[W];
    uint32_t n;
    template <int B>
    __device__ __forceinline__ void go()
    {
        for (uint32_t k = 0; k < n; ++k) {
#pragma unroll
            for (int j = 0; j < B; ++j) {
                v = r[j] * __builtin_fmaf(-v, v, v);
                if (ACC) s += __builtin_amdgcn_logf(__builtin_fabsf(__builtin_fmaf(-2.0f * r[j], v, r[j])));
            }
        }
    }
};

/* Plain steps at window positions [LO, HI), guarded past W/2 as in
 * product_range; ACC accumulates the log of the derivative. */
template <int W, bool ACC>
struct PlainRange {
    float &v;
    float &s;
    const float (&r)[W];
    uint32_t hi;
    template <int LO, int HI, bool GUARD>
    __device__ __forceinline__ void run()
    {
#pragma unroll
        for (int j = LO; j < HI; ++j) {
            if (!GUARD || j <= W / 2 || (uint32_t)j < hi) {
                v = r[j] * __builtin_fmaf(-v, v, v);
                if (ACC) s += __builtin_amdgcn_logf(__builtin_fabsf(__builtin_fmaf(-2.0f * r[j], v, r[j])));
            }
        }
    }
};

template <int W, bool ACC>
struct PlainPrefix {
    PlainRange<W, ACC> rg;
    template <int N>
    __device__ __forceinline__ void go() { rg.template run<0, N, false>(); }
};

template <int W, bool ACC>
struct PlainHead {
    PlainRange<W, ACC> rg;
    template <int N>
    __device__ __forceinline__ void go() { rg.template run<N, W, true>(); }
};

template <int W>
__device__ __forceinline__ float lambda_plain_w(float x, float y, float z,
                                                const EvalDesc &e)
{
    float r[W];
    uint32_t m[4];
    load_masks(m, e);
#pragma unroll
    for (int j = 0; j < W; ++j) r[j] = pick_mask(m, j, x, y, z, e.d);
    float v = 0.5f, s = 0.0f;
    {
        PlainFull<W, false> f{v, s, r, e.set_blocks};
        with_block_len<W>(e.B, f);
    }
    {
        PlainPrefix<W, false> f{{v, s, r, 0}};
        with_len<W>(e.set_rem, f);
    }
    if (v == 0.5f) return 0.0f / (float)e.accum;
    if (e.head_hi == e.B) {
        PlainHead<W, true> f{{v, s, r, e.B}};
        with_len<W>(e.head_lo, f);
    } else {
        plain_block<W, false>(v, s, r, e.head_lo, e.head_hi, true);
    }
    {
        PlainFull<W, true> f{v, s, r, e.acc_blocks};
        with_block_len<W>(e.B, f);
    }
    {
        PlainPrefix<W, true> f{{v, s, r, 0}};
        with_len<W>(e.acc_rem, f);
    }
    const float lam = s * kLn2f / (float)e.accum;
    return __builtin_isfinite(lam) ? lam : __builtin_nanf("");
}

/* FP64 with the reference's map ((r*v)*(1-v), separately rounded, so the
 * orbit is the IEEE double one); the derivative r(1 - 2v) only feeds the
 * log sum and is formed with one fma. The product is renormalised at the end
 * of each block and, in a 32-slot window, after its first `mid` = B/2
 * positions: at most 16 factors between renormalisations, each at most 4 in
 * magnitude while the orbit stays in [0, 1], and the same steps in either
 * window (B is then twice the 16-slot block). An orbit that escapes (a
 * sample just outside the box) can overflow between renormalisations; that
 * happens after the same steps wherever the window or launch is. */
template <int W, bool FULL, bool ACC>
__device__ __forceinline__ void fp64_block(double &v, ProductState64 &st,
                                           const double (&r)[W],
                                           const double (&m2r)[W], uint32_t lo,
                                           uint32_t hi, uint32_t mid)
{
#pragma unroll
    for (int j = 0; j < W; ++j) {
        if (in_block<W, FULL>(j, lo, hi)) {
            v = (r[j] * v) * (1.0 - v);
            if (ACC) {
                st.M *= __builtin_fabs(__builtin_fma(m2r[j], v, r[j]));
                if (W > 16 && (uint32_t)j + 1u == mid) renorm64(st);
            }
        }
    }
    if (ACC) renorm64(st);
}

/* n full FP64 blocks of B steps. */
template <int W, bool ACC>
struct Fp64Full {
    double &v;
    ProductState64 &st;
    const double (&r)[W];
    const double (&m2r)[W];
    uint32_t n;
    template <int B>
    __device__ __forceinline__ void go()
    {
        for (uint32_t k = 0; k < n; ++k) {
#pragma unroll
            for (int j = 0; j < B; ++j) {
                v = (r[j] * v) * (1.0 - v);
                if (ACC) {
                    st.M *= __builtin_fabs(__builtin_fma(m2r[j], v, r[j]));
                    if (W > 16 && j + 1 == B / 2) renorm64(st);
                }
            }
            if (ACC) renorm64(st);
        }
    }
};

/* FP64 steps at window positions [LO, HI), guarded past W/2 as in
 * product_range; the product is renormalised after position mid - 1 (a
 * 32-slot window) and at the end, as in fp64_block: exact power-of-two
 * scalings, and the final (E, M) with M in [0.5, 1) is the same wherever
 * the earlier ones fell. */
template <int W, bool ACC>
struct Fp64Range {
    double &v;
    ProductState64 &st;
    const double (&r)[W];
    const double (&m2r)[W];
    uint32_t hi, mid;
    template <int LO, int HI, bool GUARD>
    __device__ __forceinline__ void run()
    {
#pragma unroll
        for (int j = LO; j < HI; ++j) {
            if (!GUARD || j <= W / 2 || (uint32_t)j < hi) {
                v = (r[j] * v) * (1.0 - v);
                if (ACC) {
                    st.M *= __builtin_fabs(__builtin_fma(m2r[j], v, r[j]));
                    if (W > 16 && (uint32_t)j + 1u == mid) renorm64(st);
                }
            }
        }
        if (ACC) renorm64(st);
    }
};

template <int W, bool ACC>
struct Fp64Prefix {
    Fp64Range<W, ACC> rg;
    template <int N>
    __device__ __forceinline__ void go() { rg.template run<0, N, false>(); }
};

template <int W, bool ACC>
struct Fp64Head {
    Fp64Range<W, ACC> rg;
    template <int N>
    __device__ __forceinline__ void go() { rg.template run<N, W, true>(); }
};

template <int W>
__device__ __forceinline__ double lambda_fp64_w(float xf, float yf, float zf,
                                                const EvalDesc &e)
{
    double r[W], m2r[W];
    uint32_t m[4];
    load_masks(m, e);
#pragma unroll
    for (int j = 0; j < W; ++j) {
        r[j] = (double)pick_mask(m, j, xf, yf, zf, e.d);
        m2r[j] = -2.0 * r[j];
    }
    double v = 0.5;
    ProductState64 st{1.0, 0};
    const uint32_t mid = e.B / 2u;
    {
        Fp64Full<W, false> f{v, st, r, m2r, e.set_blocks};
        with_block_len<W>(e.B, f);
    }
    {
        Fp64Prefix<W, false> f{{v, st, r, m2r, 0, mid}};
        with_len<W>(e.set_rem, f);
    }
    const double off = v - 0.5;
    if (!(off <= -1e-8 || off >= 1e-8)) return 0.0 / (double)e.accum;
    if (e.head_hi == e.B) {
        Fp64Head<W, true> f{{v, st, r, m2r, e.B, mid}};
        with_len<W>(e.head_lo, f);
    } else {
        fp64_block<W, false, true>(v, st, r, m2r, e.head_lo, e.head_hi, mid);
    }
    {
        Fp64Full<W, true> f{v, st, r, m2r, e.acc_blocks};
        with_block_len<W>(e.B, f);
    }
    {
        Fp64Prefix<W, true> f{{v, st, r, m2r, 0, mid}};
        with_len<W>(e.acc_rem, f);
    }
    const double lam = ((double)st.E * kLn2 + log(st.M)) / (double)e.accum;
    return __builtin_isfinite(lam) ? lam : __builtin_nan("");
}

} /* namespace lyap */
