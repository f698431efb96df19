"""cr_pt_stats' kernel time covers the whole render, the pixels of the sky too: of a
call whose every pixel is sky it is most of what the call takes."""
import ctypes as C
import time

import pytest

pytestmark = pytest.mark.gpu


def test_sky_is_in_the_kernel_time(ctx, cfg, S):
    w, h, n = 1024, 1024, 4096
    sc = cfg.c1(width=w, height=h, size=16, sv_axis=16)
    sc.cam = cfg.camera(w, h, position=(9.0, 0.0, -0.2))   # beside the cloud, every ray misses it
    sc.setup(ctx)
    frames = (S.PushConstants * n)(*cfg.frames(n))

    def call():
        ctx.synchronize()
        t0 = time.perf_counter()
        ctx.check(ctx.lib.cr_pt_render(ctx.h, frames, n), "cr_pt_render")
        ctx.synchronize()
        return (time.perf_counter() - t0) * 1e3

    call()                                  # buffers
    ctx.pt_stats_reset()
    wall = min(call() for _ in range(3))
    st = ctx.pt_stats()
    assert st.paths == 3 * n * w * h
    kernel = st.totalKernelMs / 3
    print(f"call {wall:.2f} ms, kernel time {kernel:.2f} ms")
    assert kernel > 0.5 * wall
