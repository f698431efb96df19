"""Path-tracing launches whose work items are chunks of a pixel's frames (or of
a record's continuations): the image equals the frames rendered one call each
(one frame is never chunked), and a continuation's mean equals its samples,
taken one by one, added in order -- bit for bit."""
import numpy as np
import pytest

from gpu_util import assert_bitexact

pytestmark = pytest.mark.gpu


# 1024x1024 x 9: chunks of 4, 4 and 1 frames; 36x20 x 7: chunks of one frame,
# partial tiles; 3840x2160 x 33: more samples than one launch stores (32 + 1).
@pytest.mark.parametrize("w,h,n,dda", [(1024, 1024, 9, False), (1024, 1024, 9, True), (36, 20, 7, True),
                                       (3840, 2160, 33, False)])
def test_chunked_render_equals_single_frames(ctx, cfg, S, w, h, n, dda):
    sc = cfg.c1(width=w, height=h, size=32, sv_axis=32)
    sc.ext.bounceCap = 3
    if dda:
        sc.ext.trackingMode, sc.ext.neeMode = S.CR_TRACK_BRICK_DDA, S.CR_NEE_RATIO_TRACKING
    sc.setup(ctx)
    frames = cfg.frames(n, first=2)
    init = np.random.default_rng(n).random((h, w, 4), dtype=np.float32)
    ctx.upload_image(init)
    ctx.pt_render(frames)
    one = ctx.download_image(h, w)
    ctx.upload_image(init)
    for f in frames:
        ctx.pt_render([f])
    assert_bitexact(one, ctx.download_image(h, w), f"{w}x{h}, {n} frames in one call vs one by one")


def _next_seed(s0, s):
    """continuation_seed: the PCG hash of the recorded state and the sample index."""
    m = 0xFFFFFFFF
    state = ((s0 ^ (s * 0x9E3779B9 & m)) * 747796405 + 2891336453) & m
    word = (((state >> ((state >> 28) + 4)) ^ state) * 277803737) & m
    return ((word >> 22) ^ word) | 1


@pytest.mark.parametrize("spp", [2, 5])
def test_continuations_add_in_sample_order(ctx, cfg, S, spp):
    sc = cfg.c1(width=26, height=18, size=24, sv_axis=24)
    sc.setup(ctx)
    rec = ctx.pt_record(cfg.frames(1), 18, 26).reshape(-1, 8)   # escaped paths among the collisions
    got = ctx.pt_continue(rec, spp)
    hit = rec[:, 7] > 0.5
    assert hit.any() and not hit.all()
    acc = np.zeros((len(rec), 4), np.float32)
    for s in range(spp):
        r = rec.copy()
        if s:
            st = r.view(np.uint32)[:, 6]
            st[:] = [_next_seed(int(v), s) for v in st]
        acc = acc + ctx.pt_continue(r, 1)
    assert_bitexact(got, acc / np.float32(spp), f"{spp} continuations")
