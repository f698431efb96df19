// Allocation-free path-tracer entry point (cr_pt_render_static).
//
// cr_pt_render keeps its scratch in context buffers that it grows on demand:
// the per-frame (seed, frameCount) table, the tile list and the samples.  This
// variant keeps its frame table in a buffer of fixed size made with the context,
// like the work-queue counters, and renders whole pixels into an image the caller
// owns; tiles are claimed in raster order, which changes the schedule only (every
// pixel's arithmetic is cr_pt_render's).  It calls no hipMalloc, hipFree or
// allocating library routine.  Contexts share nothing, so their calls may overlap
// (the frame table of a GPU's contexts was one array and they raced on it; taking
// turns on it instead cost a launch's tail each, 3.6 ms a call against 1.7 at 1372x1372
// and 8 spp on three contexts).
#include "cr_runtime.h"

using namespace cr;

#define CR_CHECK_CTX(ctx) \
    do { if (!(ctx)) return CR_ERR_INVALID_ARGUMENT; } while (0)
#define CR_HIP(ctx, call, what) \
    do { hipError_t _e = (call); if (_e != hipSuccess) return hip_fail((ctx), _e, (what)); } while (0)

extern "C" {

cr_status cr_pt_render_static(cr_context* ctx, const cr_push_constants* frames, uint32_t n_frames, float* accum)
{
    CR_CHECK_CTX(ctx);
    if (!frames && n_frames) return fail(ctx, CR_ERR_INVALID_ARGUMENT, "null frames");
    if (!accum) return fail(ctx, CR_ERR_INVALID_ARGUMENT, "null accumulation image");
    if (n_frames > CR_PT_STATIC_MAX_FRAMES)
        return fail(ctx, CR_ERR_CAPACITY, "cr_pt_render_static renders at most CR_PT_STATIC_MAX_FRAMES (" +
                                              std::to_string(CR_PT_STATIC_MAX_FRAMES) + ") frames per call, got " +
                                              std::to_string(n_frames));
    if (n_frames == 0) return CR_OK;
    if (!ctx->hasGrid) return fail(ctx, CR_ERR_STATE, "no grid");
    if (ctx->W <= 0 || ctx->H <= 0) return fail(ctx, CR_ERR_STATE, "no camera set");
    if (ctx->ext.neeMode == CR_NEE_SHADOW_VOLUME && !ctx->svValid)
        return fail(ctx, CR_ERR_STATE, "shadow-volume NEE needs cr_sv_build after the last grid/shadow-volume change");
    CR_HIP(ctx, hipSetDevice(ctx->device), "hipSetDevice");

    int32_t fr[2 * CR_PT_STATIC_MAX_FRAMES];
    for (uint32_t i = 0; i < n_frames; i++) {
        fr[2 * i] = frames[i].seed;
        fr[2 * i + 1] = (int32_t)frames[i].frameCount;
    }
    int32_t* dFrames = ctx->staticFrames;
    // stream order: the copy waits for any earlier kernel that still reads the table
    CR_HIP(ctx, hipMemcpyAsync(dFrames, fr, (size_t)n_frames * 8, hipMemcpyHostToDevice, ctx->stream), "copy frames");
    CR_HIP(ctx, hipStreamSynchronize(ctx->stream), "sync frames");
    CR_HIP(ctx, zero_async(ctx->dQueue, PT_QUEUE_WORDS * 4, ctx->stream), "clear queue");

    PTArgs a;
    fill_job_args(a, ctx->grid, ctx->sv, ctx->svDimsBuilt, ctx->cam, ctx->cloud, ctx->params, ctx->svp, ctx->ext,
                  dFrames, n_frames, accum, ctx->W, ctx->H, ctx->ptTileLog2W);
    a.queue = ctx->dQueue;
    a.counters = nullptr;
    const DeviceGrid& g = ctx->grid;
    int blocks = ctx->numCUs * pt_blocks_per_cu(g.dtype, g.layout, ctx->ext.trackingMode, ctx->ext.neeMode, n_frames);
    const uint32_t needed = (a.totalIdx + 255u) / 256u;
    if ((uint32_t)blocks > needed) blocks = (int)needed;
    CR_HIP(ctx, launch_pt(a, g.dtype, g.layout, blocks, ctx->numCUs, ctx->stream), "path tracer kernel");
    return CR_OK;
}

} // extern "C"
