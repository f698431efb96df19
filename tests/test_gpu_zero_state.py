"""The generator's fixed point in the path tracer: a frame whose seed is 0 (and, in
every frame, pixel 0) starts from the state 0, draws only 0 and so makes infinite
free flights.  The cloud is hundreds of mean free paths deep, so that a large but
finite flight would end in it."""
import ctypes as C

import numpy as np
import pytest

from gpu_util import assert_bitexact, oracle_scene_from_ctx
from test_zz_no_alloc import DeviceImage

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tracking", ["CR_TRACK_GLOBAL_MAJORANT", "CR_TRACK_BRICK_DDA"])
@pytest.mark.parametrize("nee", ["CR_NEE_SHADOW_VOLUME", "CR_NEE_RATIO_TRACKING"])
def test_zero_state(ctx, cfg, S, O, pkg, tracking, nee):
    w, h = 20, 14
    sc = cfg.c1(width=w, height=h, size=24, sv_axis=24)
    sc.density_scaling *= 12.0
    sc.cam = cfg.camera(w, h, position=(0.0, 0.0, 0.3))   # inside: every pixel's ray crosses the cloud
    sc.ext = cfg.render_ext(albedo=0.9, bounce_cap=16, sky=cfg.SKY, nee=getattr(S, nee), tracking=getattr(S, tracking))
    cloud, svp = sc.setup(ctx)
    s, _, _ = oracle_scene_from_ctx(O, ctx, sc.cam, sc.params, svp, sc.ext)
    frames = cfg.frames(18)         # the static call below: more frames than the few-frame kernel takes
    for k in (0, 5):
        frames[k].seed = 0
    ref, cnt = O.pt_render(s, frames)
    ctx.pt_stats_reset()
    ctx.pt_render(frames)
    assert_bitexact(ctx.download_image(h, w), ref, "image")
    st = ctx.pt_stats()
    assert (st.paths, st.vertices, st.lookups) == (cnt.paths, cnt.vertices, cnt.lookups)
    img = DeviceImage(np.zeros((h, w, 4), np.float32))
    arr = (S.PushConstants * len(frames))(*frames)
    ctx.check(ctx.lib.cr_pt_render_static(ctx.h, arr, len(frames), C.c_void_p(img.ptr.value)), "cr_pt_render_static")
    ctx.synchronize()
    assert_bitexact(img.download((h, w, 4)), ref, "static image")
    img.free()
