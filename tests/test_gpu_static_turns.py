"""cr_pt_render_static on two contexts whose streams run at the same time: calls
that follow each other without a wait give the images of cr_pt_render."""
import ctypes as C

import numpy as np
import pytest

from gpu_util import assert_bitexact
from test_zz_no_alloc import DeviceImage

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,n", [(64, 48, 2), (1024, 768, 6), (256, 256, 40)])
def test_overlapping_static_renders(pkg, cfg, S, w, h, n):
    zero = np.zeros((h, w, 4), np.float32)
    jobs = []
    for k in range(2):
        ctx = pkg.Context(0)
        sc = cfg.c1(width=w, height=h, size=32, sv_axis=32)
        sc.setup(ctx)
        frames = cfg.frames(n, first=1 + 100 * k)
        jobs.append((ctx, frames, (S.PushConstants * n)(*frames),
                     DeviceImage(zero)))
    for _ in range(2):
        for ctx, _, arr, img in jobs:
            ctx.check(ctx.lib.cr_pt_render_static(ctx.h, arr, n, C.c_void_p(img.ptr.value)), "cr_pt_render_static")
    for ctx, _, _, _ in jobs:
        ctx.check(ctx.lib.cr_synchronize(ctx.h), "cr_synchronize")
    for ctx, frames, _, img in jobs:
        ctx.upload_image(zero)
        ctx.pt_render(frames)
        ctx.pt_render(frames)
        assert_bitexact(img.download((h, w, 4)), ctx.download_image(h, w), f"{w}x{h}, {n} frames")
        img.free()
