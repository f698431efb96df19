"""Renders of several frames in one call: their tiles are listed by squares of
64x64 pixels, tiles and pixels that miss the cloud are left to the listing
kernel.  Image and path counts equal those of the frames rendered one call each
(a single frame takes all tiles in raster order), bit for bit."""
import numpy as np
import pytest

from gpu_util import assert_bitexact

pytestmark = pytest.mark.gpu


# (2, 2): one partial tile; (64, 64) one square; (66, 62): squares of one column
# and a missing row; (520, 70): 18 squares for 8 parts; z = -2: most tiles miss
# the box; x = 9: all of them do.
@pytest.mark.parametrize("w,h", [(2, 2), (64, 64), (66, 62), (520, 70)])
@pytest.mark.parametrize("pos", [(0.0, 0.0, -0.2), (0.1, 0.0, -2.0), (9.0, 0.0, -0.2)])
def test_listed_render_equals_single_frames(ctx, cfg, S, w, h, pos):
    sc = cfg.c1(width=w, height=h, size=32, sv_axis=32)
    sc.cam = cfg.camera(w, h, position=pos)
    sc.setup(ctx)
    frames = cfg.frames(3, first=1)
    init = np.random.default_rng(w + h).random((h, w, 4), dtype=np.float32)

    def render(calls):
        ctx.upload_image(init)
        ctx.pt_stats_reset()
        for c in calls:
            ctx.pt_render(c)
        st = ctx.pt_stats()
        return ctx.download_image(h, w), (st.paths, st.vertices, st.lookups, st.svLookups)

    one, n_one = render([frames])
    each, n_each = render([[f] for f in frames])
    assert_bitexact(one, each, f"{w}x{h} from {pos}")
    assert n_one == n_each and n_one[0] == 3 * w * h
