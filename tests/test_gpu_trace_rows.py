"""The photon tracers against the oracle where they can go wrong: walks of many
rounds, paths without an interaction, more records than the first guess has
room for, more paths than one launch takes, truncation, waves with few paths,
and the generator's fixed point (seed 0)."""
import pytest

from gpu_util import oracle_scene_from_ctx
from test_gpu_ppm import oracle_map, setup as ppm_setup

pytestmark = pytest.mark.gpu

# paths, radius, albedo, interactions, density factor, max_beams, seed
CASES = {
    "grow": (700, 0.3, 1.0, 64, 30.0, 1 << 20, 38),        # tens of interactions per path
    "two_launches": (264000, 0.9, 0.0, 8, 0.06, 1 << 20, 5),
    "long_walks": (60, 0.05, 0.9, 16, 12.0, 1 << 20, 7),   # hundreds of steps per walk
    "cut": (900, 0.01, 0.9, 64, 1.0, 5000, 38),
    "one": (1, 0.02, 0.9, 1, 1.0, 1 << 20, 3),
    "seed0": (37, 0.02, 0.9, 64, 1.0, 1 << 20, 0),
    "none": (50, 0.02, 0.9, 0, 1.0, 1 << 20, 3),
}


@pytest.mark.parametrize("name", list(CASES))
def test_trace_beams_rows(ctx, cfg, S, O, name):
    paths, radius, albedo, inter, dense, most, seed = CASES[name]
    sc = cfg.c1(width=32, height=32, size=40, sv_axis=32)
    if name in ("grow", "cut"):
        sc.storage, sc.grid_layout = S.CR_DTYPE_F16, S.CR_GRID_BRICK4
    sc.density_scaling *= dense
    cloud, svp = sc.setup(ctx, build_sv=False)
    p = cfg.beam_params(paths, seed=seed, radius=radius, albedo=albedo, max_interactions=inter)
    nb, nd = ctx.trace_beams(p, most)
    s, _, _ = oracle_scene_from_ctx(O, ctx, sc.cam, sc.params, svp, sc.ext, with_sv=False)
    rb, rd, rnb, rnd = O.trace_beams(s, p, most)
    assert (nb, nd) == (rnb, rnd)
    if name == "grow":
        assert nd > 8 * paths + 1024
    if nb:
        gb, gd = ctx.download_beams()
        assert bytes(gb) == bytes(rb)[:nb * 48], "beams differ"
        assert bytes(gd) == bytes(rd)[:nd * 80], "beam data differ"
    else:
        assert name == "none"


@pytest.mark.parametrize("paths,seed,dense", [(1, 38, 1.0), (37, 0, 1.0), (100, 5, 30.0), (5000, 9, 1.0), (40001, 3, 0.3)])
def test_ppm_trace_rows(ctx, cfg, S, O, pkg, paths, seed, dense):
    sc, cloud, svp, pm, p = ppm_setup(ctx, cfg, S, pkg)
    cloud.densityScaling *= dense
    ctx.set_cloud(cloud)
    ctx.sv_build()
    p.numPaths = paths
    n = ctx.ppm_trace(seed, p)
    _, photons, nd = ctx.ppm_download()
    _, rn, _, _, rsorted = oracle_map(O, ctx, sc, svp, pm, p, seed)
    assert nd == n == rn
    assert bytes(photons)[:48 * n] == bytes(rsorted)[:48 * n], "photon grid differs"
    if dense > 1.0:
        assert n > 8 * paths + 16 * (paths // 2 + 64)   # more chunks than the first guess
