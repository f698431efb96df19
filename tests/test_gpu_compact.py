"""The learned render's compaction in one pass: record counts around its
workgroups of 4096, one call against single frames, and escaped pixels against
their records."""
import numpy as np
import pytest

from gpu_util import assert_bitexact

pytestmark = pytest.mark.gpu


# 4, 4096, 4096 + 128, and 3 x 4104 records
@pytest.mark.parametrize("w,h,n", [(2, 2, 1), (64, 64, 1), (66, 64, 1), (76, 54, 3)])
def test_one_pass_compaction(ctx, cfg, S, w, h, n):
    sc = cfg.c1(width=w, height=h, size=32, sv_axis=32)
    sc.ext = cfg.render_ext(albedo=0.9, bounce_cap=16, sky=cfg.SKY, nee=S.CR_NEE_RATIO_TRACKING)
    sc.setup(ctx)
    ctx.mlp_init(3)
    frames = cfg.frames(n)
    ctx.clear_image()
    ctx.learn_render(frames)
    once = ctx.download_image(h, w)
    ctx.clear_image()
    for f in frames:
        ctx.learn_render([f])
    assert_bitexact(ctx.download_image(h, w), once, f"{n} frames of {w}x{h}")
    # the pixels whose paths escaped show the record's radiance
    rec = ctx.pt_record(frames, h, w)
    if n == 1:
        out = rec[0][..., 7] <= 0.5
        assert_bitexact(once[out], rec[0][..., :4][out], "escaped pixels")
        assert w == 2 or (out.any() and not out.all())
