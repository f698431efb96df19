"""Density and shadow-volume lookups: launch-constant divisors (powers of two, any
others, and ones too large for the residual form) and grids whose rows are read
in pairs of voxels (rows of one, two and an odd number), against the oracle."""
import numpy as np
import pytest

from gpu_util import assert_bitexact, oracle_scene_from_ctx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,scale", [((16, 16, 16), 1.0), ((1, 6, 5), 1.0), ((2, 3, 4), 0.3), ((33, 18, 7), 1.7),
                                        ((21, 30, 17), 2.0 ** 70)])
@pytest.mark.parametrize("half", [False, True])
def test_lookups_bitexact(ctx, cfg, S, O, dims, scale, half):
    nx, ny, nz = dims
    w, h = 24, 18
    sc = cfg.c1(width=w, height=h, size=16, sv_axis=19)
    sc.cam = cfg.camera(w, h, position=(0.0, 0.0, -0.2 * scale))
    sc.setup(ctx, build_sv=False)
    grid = (np.random.default_rng(nx).random((nz, ny, nx)) ** 2).astype(np.float32)
    ctx.upload_grid(grid, 1.0 / max(dims), storage=S.CR_DTYPE_F16 if half else S.CR_DTYPE_F32)
    cloud = ctx.cloud()
    for k in range(3):
        cloud.bounds[0][k] *= scale
        cloud.bounds[1][k] *= scale
    cloud.densityScaling /= scale
    ctx.set_cloud(cloud)
    for light in ((0.3, -1.0, 0.4), (0.0, -1.0, 0.0)):
        svp = cfg.shadow_volume(cloud, light, 19)
        ctx.set_shadow_volume(svp)
        ctx.sv_build()
        s, _, sv = oracle_scene_from_ctx(O, ctx, sc.cam, sc.params, svp, sc.ext)
        assert_bitexact(sv, O.sv_build(s), f"shadow volume, light {light}")
        frames = cfg.frames(2)
        ctx.clear_image()
        ctx.pt_render(frames)
        ref, _ = O.pt_render(s, frames)
        # Pixel 0 is left out: its seed is 0 and so are all its draws, and the
        # path tracer's flights take -log 0 as 88 where the oracle's are infinite
        # (it shows where a ray crosses more than 88 mean free paths).
        img = ctx.download_image(h, w).reshape(-1, 4)[1:]
        assert_bitexact(img, ref.reshape(-1, 4)[1:], f"image, light {light}")


# 320 x 511 columns are summed in two passes, 320 x 512 in one; 17 texels: one
# more than the second pass fetches together
@pytest.mark.parametrize("dims", [(2, 2, 2), (65, 5, 17), (320, 511, 3), (320, 512, 3), (9, 7, 33)])
def test_shadow_volume_passes(ctx, cfg, S, O, dims):
    sc = cfg.c1(width=4, height=4, size=24, sv_axis=33)
    sc.ext = cfg.render_ext(albedo=0.9, bounce_cap=16, sky=cfg.SKY, sv_dims=dims)
    cloud, svp = sc.setup(ctx)
    s, _, sv = oracle_scene_from_ctx(O, ctx, sc.cam, sc.params, svp, sc.ext)
    assert_bitexact(sv, O.sv_build(s), f"shadow volume of {dims}")
