"""Renders of whole pixels: single frames, and the static entry point with few and
with many frames, on images of up to a wave per SIMD (256x256 on 256 CUs), one
column of tiles more, and partial tiles, against the same frames in work items of a
few frames."""
import ctypes as C

import numpy as np
import pytest

from gpu_util import assert_bitexact
from test_zz_no_alloc import DeviceImage

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(2, 2), (66, 62), (256, 256), (264, 256), (258, 250)])
@pytest.mark.parametrize("n", [2, 16, 17])
def test_whole_pixels(ctx, cfg, S, w, h, n):
    sc = cfg.c1(width=w, height=h, size=24, sv_axis=24)
    sc.setup(ctx)
    frames = cfg.frames(n, first=1)
    init = np.random.default_rng(w + h).random((h, w, 4), dtype=np.float32)
    ctx.upload_image(init)
    ctx.pt_render(frames)
    ref = ctx.download_image(h, w)
    ctx.upload_image(init)
    for f in frames:
        ctx.pt_render([f])
    assert_bitexact(ctx.download_image(h, w), ref, "frame by frame")
    img = DeviceImage(init)
    arr = (S.PushConstants * n)(*frames)
    ctx.check(ctx.lib.cr_pt_render_static(ctx.h, arr, n, C.c_void_p(img.ptr.value)), "cr_pt_render_static")
    ctx.synchronize()
    assert_bitexact(img.download((h, w, 4)), ref, "static")
    img.free()
