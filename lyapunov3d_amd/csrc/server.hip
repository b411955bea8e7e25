/*
 * server.hip - the serving loop's device side: continuous batching of view
 * and volume requests on one GPU.
 *
 * The scheduler (serve_core.cpp) decides what each launch carries; this file
 * runs the launches. Every slot owns a context of its own (stream, launch
 * buffers, counters), so launches of different slots overlap on the device
 * and a launch that is finishing its long rays shares the CUs with the next
 * one. A mixed slot runs its views in one launch sequence and then its
 * volumes' slabs in the volume kernels (lyap_run_batch's path). With LYAP_SERVER_SEPARATE_VOLUMES (or when the volume
 * precision differs from the views') render slots take views only and
 * volume slots run slabs in the volume kernels.
 *
 * The reference renders one view per launch from an interactive loop
 * (lyap_interactive.cu:711) and one volume per process (lyap_calculate.cu:72);
 * it has no request queue.
 */
#include <chrono>
#include <cstring>
#include <thread>
#include <vector>

#include "internal.hpp"
#include "serve_core.hpp"

using namespace lyap;
using namespace lyap::serve;

namespace {

struct HipSlot {
    lyap_ctx *ctx = nullptr;
    int kind = SLOT_MIXED;
    RenderSlot *rs = nullptr;
    hipEvent_t start = nullptr, end = nullptr;
    /* pinned: the lambda evaluations of the launch's views */
    uint64_t *host_evals = nullptr;   /* kEvalSlots counts */
    /* FP64 re-evaluations of each slab: on the device and pinned */
    uint32_t *reeval = nullptr, *host_reeval = nullptr;
    unsigned nblocks = 0;
    bool has_views = false;
    uint64_t voxels = 0;
};

class HipBackend final : public ServeBackend {
public:
    HipBackend(lyap_ctx *owner, const LyapServerConfig &cfg)
        : owner_(owner), cfg_(cfg), t0_(std::chrono::steady_clock::now())
    {
    }

    /* Creates the slots' contexts, events and pinned result words. */
    int init(const std::vector<int> &kinds)
    {
        slots_.resize(kinds.size());
        for (size_t i = 0; i < kinds.size(); ++i) {
            HipSlot &sl = slots_[i];
            sl.kind = kinds[i];
            int rc = lyap_create(&sl.ctx, owner_->device, 0);
            if (rc) return fail(owner_, rc, "server slot context: %s", lyap_strerror(rc));
            const size_t reeval_bytes = kMaxSlabs * sizeof(uint32_t);
            if (hipEventCreate(&sl.start) != hipSuccess || hipEventCreate(&sl.end) != hipSuccess ||
                hipHostMalloc((void **)&sl.host_evals, kEvalBytes, hipHostMallocDefault) !=
                    hipSuccess ||
                hipHostMalloc((void **)&sl.host_reeval, reeval_bytes, hipHostMallocDefault) != hipSuccess)
                return fail(owner_, LYAP_ERR_DEVICE, "server slot set-up failed");
            std::memset(sl.host_evals, 0, kEvalBytes);
            std::memset(sl.host_reeval, 0, reeval_bytes);
            if (sl.kind != SLOT_VOLUME) sl.rs = render_slot_create();
            if (sl.kind != SLOT_RENDER && has_rule(cfg_.vol_mode)) {
                /* re-evaluation list for the largest slab (256 x 256 x 256) up
                 * front, so a slab never reallocates while others run */
                rc = ensure_reeval_list(sl.ctx, 256u * 256u * 256u);
                void *p = nullptr;
                if (rc == LYAP_OK) rc = ctx_alloc(sl.ctx, &p, reeval_bytes);
                if (rc) {
                    owner_->last_error = sl.ctx->last_error;
                    return rc;
                }
                sl.reeval = (uint32_t *)p;
            }
        }
        return LYAP_OK;
    }

    ~HipBackend() override
    {
        sync_all();
        for (auto &sl : slots_) {
            if (sl.rs) render_slot_destroy(sl.ctx, sl.rs);
            if (sl.start) (void)hipEventDestroy(sl.start);
            if (sl.end) (void)hipEventDestroy(sl.end);
            if (sl.host_evals) (void)hipHostFree(sl.host_evals);
            if (sl.host_reeval) (void)hipHostFree(sl.host_reeval);
            if (sl.ctx) lyap_destroy(sl.ctx);
        }
    }

    double now_ms() override
    {
        return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0_).count();
    }

    int alloc(size_t bytes, void **out) override { return ctx_alloc(owner_, out, bytes); }

    void release(void *p) override
    {
        sync_all();   /* a free waits for the device anyway */
        ctx_free(owner_, p);
    }

    int launch(unsigned i, const SlotLaunch &l) override
    {
        HipSlot &sl = slots_[i];
        const int rc = launch_on(sl, l);
        if (rc) owner_->last_error = sl.ctx->last_error;
        return rc;
    }

    int query(unsigned i, LaunchResult *res) override
    {
        HipSlot &sl = slots_[i];
        const hipError_t q = hipEventQuery(sl.end);
        if (q == hipErrorNotReady) return LYAP_ERR_PENDING;
        if (q != hipSuccess) return fail(owner_, LYAP_ERR_DEVICE, "server launch: %s", hipGetErrorString(q));
        float ms = 0.0f;
        res->ms = hipEventElapsedTime(&ms, sl.start, sl.end) == hipSuccess ? (double)ms : -1.0;
        res->evals = sl.voxels + (sl.has_views ? sum_evals(sl.host_evals) : 0u);
        for (unsigned b = 0; b < sl.nblocks && b < kMaxSlabs; ++b)
            res->reeval[b] = sl.host_reeval[b];
        return LYAP_OK;
    }

    void idle() override { std::this_thread::sleep_for(std::chrono::microseconds(20)); }

    int error(int code, const char *msg) override { return fail(owner_, code, "%s", msg); }

private:
    void sync_all()
    {
        for (auto &sl : slots_)
            if (sl.ctx) (void)hipStreamSynchronize(sl.ctx->stream);
    }

    int launch_on(HipSlot &sl, const SlotLaunch &l)
    {
        sl.nblocks = (unsigned)l.blocks.size();
        sl.has_views = !l.views.empty();
        sl.voxels = l.voxels;
        LYAP_HIP(sl.ctx, hipEventRecord(sl.start, sl.ctx->stream));
        if (sl.has_views) {
            int rc = render_slot_launch(sl.ctx, sl.rs, l.views.data(), l.begin.data(), l.count.data(),
                                        (unsigned)l.views.size(), cfg_.mode, owner_->tuned);
            if (rc) return rc;
            LYAP_HIP(sl.ctx, hipMemcpyAsync(sl.host_evals, render_slot_counters(sl.rs), kEvalBytes,
                                            hipMemcpyDeviceToHost, sl.ctx->stream));
        }
        if (sl.nblocks) {
            int rc = launch_blocks(sl.ctx, l.blocks.data(), sl.nblocks, cfg_.vol_mode, sl.reeval);
            if (rc) return rc;
            if (has_rule(cfg_.vol_mode))
                LYAP_HIP(sl.ctx, hipMemcpyAsync(sl.host_reeval, sl.reeval, sl.nblocks * sizeof(uint32_t),
                                                hipMemcpyDeviceToHost, sl.ctx->stream));
        }
        LYAP_HIP(sl.ctx, hipEventRecord(sl.end, sl.ctx->stream));
        return LYAP_OK;
    }

    lyap_ctx *owner_;                  /* owner of resident outputs */
    LyapServerConfig cfg_;
    std::chrono::steady_clock::time_point t0_;
    std::vector<HipSlot> slots_;
};

} /* namespace */

extern "C" int lyap_server_create(lyap_ctx *ctx, const LyapServerConfig *cfg_in, lyap_server **out)
{
    if (!out) return LYAP_ERR_INVALID_ARGUMENT;
    *out = nullptr;
    if (!ctx) return LYAP_ERR_INVALID_ARGUMENT;
    LyapServerConfig cfg;
    std::string why;
    int rc = check_config(cfg_in, &cfg, &why);
    if (rc) return fail(ctx, rc, "%s", why.c_str());
    HipBackend *dev = new HipBackend(ctx, cfg);
    rc = dev->init(slot_kinds(cfg));
    if (rc) {
        delete dev;
        return rc;
    }
    *out = server_new(cfg, dev);
    return LYAP_OK;
}
