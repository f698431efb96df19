"""Optional scratch on a device that is nearly full: the samples a context keeps make
way for what a later call cannot do without, a render with less room for samples
takes more launches, and images stay the same."""
import ctypes as C

import pytest

from gpu_util import assert_bitexact

pytestmark = pytest.mark.gpu
GIB = 1 << 30


class Full:
    """Device memory taken but for `left` bytes."""

    def __init__(self, left):
        self.hip = C.CDLL("libamdhip64.so.7")
        self.held = []
        size = 64 * GIB
        while self.free() > left + (256 << 20) and size >= 256 << 20:
            p = C.c_void_p()
            if self.hip.hipMalloc(C.byref(p), C.c_size_t(min(self.free() - left, size))) == 0:
                self.held.append(p)
            else:
                size //= 2      # no piece of that size is free

    def free(self):
        f, t = C.c_size_t(), C.c_size_t()
        assert self.hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    def release(self):
        for p in self.held:
            assert self.hip.hipFree(p) == 0
        self.held = []


@pytest.mark.parametrize("batch", [False, True])
def test_samples_make_way(pkg, cfg, S, batch):
    w = h = 1024
    frames = cfg.frames(256, first=1)       # 4 GiB of samples
    ctx = pkg.Context(0)
    sc = cfg.c1(width=w, height=h, size=32, sv_axis=32)
    sc.cam = cfg.camera(w, h, position=(0.0, 0.0, -3.0))
    sc.ext = cfg.render_ext(albedo=0.9, bounce_cap=4, sky=cfg.SKY, nee=S.CR_NEE_NONE)

    def render():
        if batch:
            ctx.batch_clear_images()
            ctx.batch_render()
            return ctx.batch_download(0)
        ctx.clear_image()
        ctx.pt_render(frames)
        return ctx.download_image(h, w)

    sc.setup(ctx, build_sv=False)
    if batch:
        ctx.batch_add(frames)
    ref = render()
    full = Full(3 * GIB)
    try:
        # 4 GiB of voxels: more than is left, less than is left and the samples
        ctx.generate_fbm(cfg.fbm((1024, 1024, 1024), 1.0 / 1024, octaves=1), S.CR_DTYPE_F32)
        assert full.free() < 4 * GIB
        if not batch:
            sc.fbm.size[:] = (64, 64, 64)
            sc.fbm.voxelSize = 1.0 / 64
            sc.setup(ctx, build_sv=False)   # another cloud
            more = Full(2 * GIB)
            full.held += more.held
        few = render()
    finally:
        full.release()
    if batch:
        assert_bitexact(few, ref, "batch image")
    else:
        assert_bitexact(few, render(), "image")
    ctx.close()


def test_no_room_for_samples(pkg, cfg, S):
    """Room for less than two frames: whole pixels, from the list of the tiles."""
    w = h = 8192
    frames = cfg.frames(20, first=1)
    ctx = pkg.Context(0)
    sc = cfg.c1(width=w, height=h, size=32, sv_axis=32)
    sc.cam = cfg.camera(w, h, position=(0.0, 0.0, -3.0))
    sc.setup(ctx)
    full = Full(3 * GIB // 2)               # two frames of samples are 2 GiB
    try:
        ctx.pt_render(frames)
        whole = ctx.download_image(h, w)
    finally:
        full.release()
    ctx.clear_image()
    ctx.pt_render(frames)
    assert_bitexact(whole, ctx.download_image(h, w), "image")
    ctx.close()
