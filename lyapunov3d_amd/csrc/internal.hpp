/*
 * internal.hpp - host-side state shared by the library's translation units.
 */
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdio>
#include <string>
#include <unordered_map>
#include <vector>

#include "lyap.h"
#include "lyap_device.hpp"

struct lyap_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    size_t budget = 0;          /* 0: no cap */
    size_t in_use = 0;          /* bytes the library allocated */
    std::string last_error;
    std::unordered_map<void *, size_t> allocations;

    /* scratch: counters of the FP64 re-evaluation list's parts, then (word
     * kReevalWords) the entries of the last list */
    uint32_t *counters = nullptr;
    uint32_t *reeval_list = nullptr;   /* voxel indices for the FP64 pass */
    size_t reeval_cap = 0;             /* entries */
    bool has_reevaluated = false;      /* the last volume call had a rule, and so a list */

    /* the render path's launch resources (render.hip) */
    void *render_res = nullptr;
    uint32_t *last_counters = nullptr; /* counters of the last render launch */
    uint64_t last_voxels = 0;          /* voxels of the last batch's blocks */

    LyapTuning tuned{};                /* autotuner's choice, zero = unset */
    void *debug_wave_log = nullptr;    /* per-wave render record, when set */
    int num_cus = 0;

    /* kernel timing: event pairs around render launches, reused */
    bool timing = false;
    std::vector<hipEvent_t> timing_events;
    size_t timing_used = 0;            /* events recorded since the last collect */
};

namespace lyap {

int fail(lyap_ctx *ctx, int code, const char *fmt, ...);

/* Allocation through the context's budget. */
int ctx_alloc(lyap_ctx *ctx, void **ptr, size_t bytes);
void ctx_free(lyap_ctx *ctx, void *ptr);

/* The FP64 re-evaluation list is kReevalParts parts with a counter each on a
 * 128-byte line. A device-scope atomic takes 10 to 20 ns on its address, one
 * after the other: with one counter the 29,600 waves of a 154 x 184 x 67
 * volume at 464 iterations queued for 343 us (72 us with these). */
constexpr uint32_t kReevalParts = 64;
constexpr uint32_t kReevalStride = 32;            /* words */
constexpr uint32_t kReevalWords = kReevalParts * kReevalStride;
/* Whether the mode re-evaluates voxels in FP64. */
inline bool has_rule(const LyapVolumeMode &m)
{
    return m.precision == LYAP_PREC_PRODUCT && (m.fp64_margin > 0.0f || m.converge_tau > 0.0f);
}

int ensure_reeval_list(lyap_ctx *ctx, size_t entries);

/* Records the next timing event on the context's stream (no-op when timing
 * is off). */
int timing_mark(lyap_ctx *ctx);

/* Launchers in the kernel translation units. */
int launch_zero_u32(lyap_ctx *ctx, uint32_t *p, uint32_t n);

int launch_volume(lyap_ctx *ctx, float *out, const EvalDesc &e,
                  const float lo[3], const float hi[3], unsigned nx,
                  unsigned ny, unsigned nz, const float *xyz, size_t npoints,
                  const LyapVolumeMode &mode);

void free_render_resources(lyap_ctx *ctx);

/* z slices [z_begin, z_end) of a grid. With a rule the voxels re-evaluated are
 * counted in *total (device memory; null: the context's word). */
int launch_volume_slab(lyap_ctx *ctx, float *out, const EvalDesc &e,
                       const float lo[3], const float hi[3], unsigned nx,
                       unsigned ny, unsigned nz, unsigned z_begin, unsigned z_end,
                       const float *xyz, size_t npoints, const LyapVolumeMode &mode,
                       uint32_t *total = nullptr);

/* The allocation-free volume path: entries of its scratch list (16 MiB). */
constexpr uint32_t kNoAllocListCap = 1u << 22;
/* Looks up the scratch array's address on `device` (current) once per
 * device; lyap_create calls it. */
int noalloc_scratch_setup(int device);
int launch_volume_noalloc(lyap_ctx *ctx, float *out, const EvalDesc &e, const float lo[3],
                          const float hi[3], unsigned nx, unsigned ny, unsigned nz,
                          const LyapVolumeMode &mode);

int launch_points_halves(lyap_ctx *ctx, float *lam, float *h1, float *h2, const EvalDesc &e,
                         const float *xyz, size_t n);

/* Server launch slots (render.hip). */
struct RenderSlot;
RenderSlot *render_slot_create();
void render_slot_destroy(lyap_ctx *ctx, RenderSlot *slot);
/* Lambda evaluations of a launch (rays' algorithmic samples) are counted in kEvalSlots 64-bit words, one per 128-byte line, and
 * added up by whoever reads them: device-scope atomics on one address take
 * about 20 ns each, one after the other, and with one word the 5,000 waves of
 * a 512 x 512 frame's refinement ended in a queue (116 us; 112 us with
 * these). */
constexpr uint32_t kEvalSlots = 64;
constexpr uint32_t kEvalStride = 16;              /* 64-bit words per line */
constexpr size_t kEvalBytes = (size_t)kEvalSlots * kEvalStride * sizeof(uint64_t);
inline uint64_t sum_evals(const uint64_t *words)
{
    uint64_t n = 0;
    for (uint32_t k = 0; k < kEvalSlots; ++k) n += words[k * kEvalStride];
    return n;
}
/* The slot's counter block, which begins with those words. */
const uint32_t *render_slot_counters(const RenderSlot *slot);
int render_slot_launch(lyap_ctx *ctx, RenderSlot *slot, const LyapView *views,
                       const uint32_t *ray_begin, const uint32_t *ray_count, unsigned n,
                       const LyapRenderMode &mode, const LyapTuning &tune);

/* Volume blocks through the volume kernels (render.hip). */
int launch_blocks(lyap_ctx *ctx, const LyapVolumeBlock *blocks, unsigned n, const LyapVolumeMode &vmode,
                  uint32_t *totals);

int launch_render(lyap_ctx *ctx, LyapRGBA *rgba, LyapPoint *points,
                  const LyapCam &cam, const LyapParams &prm, const EvalDesc &e,
                  const LyapLight *lights, unsigned num_lights, unsigned w,
                  unsigned h, float *depth, float *lambda, uint32_t *evals,
                  const LyapRenderMode &mode);

} /* namespace lyap */

#define LYAP_HIP(ctx, call)                                                   \
    do {                                                                      \
        hipError_t _e = (call);                                               \
        if (_e != hipSuccess)                                                 \
            return lyap::fail((ctx), LYAP_ERR_DEVICE, "%s: %s (%s:%d)", #call, \
                              hipGetErrorString(_e), __FILE__, __LINE__);     \
    } while (0)
