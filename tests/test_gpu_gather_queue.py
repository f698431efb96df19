"""The gather's deferred beam tests against the oracle: a tree deep enough that
the traversal stack leaves LDS, with more hit leaves per ray than the queues
hold, and ragged images whose waves are partly outside."""
import numpy as np
import pytest

from gpu_util import assert_bitexact, oracle_scene_from_ctx

pytestmark = pytest.mark.gpu


def chain_beams(S, zeros, radius):
    """Two beams at each of the 30 Morton codes 2^k and `zeros` at code 0: the
    hierarchy is a chain of 30 nodes whose right children are inner nodes, so
    a ray that hits every box stacks one entry per level."""
    c = [(0.0, 0.0, 0.0)] * zeros
    for j in range(1, 11):
        for axis in range(3):
            p = [0.0, 0.0, 0.0]
            p[axis] = 2.0 ** -j
            c += [tuple(p)] * 2
    c = np.array(c, np.float32) + np.array([-0.5, -0.5, 0.0], np.float32)
    n = len(c)
    beams = (S.PhotonBeam * n)()
    f = np.frombuffer(beams, np.float32).reshape(n, 12)
    u = np.frombuffer(beams, np.uint32).reshape(n, 12)
    # directions differ per beam, so every one adds its own term; each keeps
    # its centroid (start and end are mirrored about it)
    rng = np.random.default_rng(n)
    d = rng.normal(size=(n, 3))
    h = (0.25 * d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    f[:, 0:3] = c - h
    f[:, 4:7] = c + h
    f[:, 7] = radius
    u[:, 8] = np.arange(n) % 4
    data = (S.PhotonBeamData * 4)()
    for i in range(4):
        data[i].power[:] = (1.0, 0.5, 0.25, 1.0)
        data[i].trDistances[:] = tuple(np.linspace(0.05, 0.6, 16) * (i + 1) / 2)
    return beams, data


@pytest.mark.parametrize("zeros,w,h", [(2, 46, 30), (700, 18, 10)])
def test_gather_of_a_chain(ctx, cfg, S, O, zeros, w, h):
    sc = cfg.c1(width=w, height=h, size=32, sv_axis=32)
    cloud, _ = sc.setup(ctx, build_sv=False)
    svp = cfg.shadow_volume(cloud, tuple(sc.cam.forward), 32)
    ctx.set_shadow_volume(svp)
    ctx.sv_build()
    beams, data = chain_beams(S, zeros, 0.7)
    n = len(beams)
    ctx.upload_beams(beams, data)
    ctx.lbvh_build()
    ctx.clear_image()
    fr = cfg.frames(2)
    g0 = ctx.gather_stats()
    ctx.gather(fr, S.GatherExt(0, 0, 0.9, 0))
    g1 = ctx.gather_stats()
    gpu = ctx.download_image(h, w)
    keys, perm, nodes = ctx.lbvh_download()
    assert len(set(keys.tolist())) >= 28                    # the chain's codes (rounding may merge the finest)
    assert g1.nodesVisited - g0.nodesVisited > 30 * (g1.rays - g0.rays)
    sorted_beams = (S.PhotonBeam * n)(*[beams[int(i)] for i in perm])
    for i in range(n):
        sorted_beams[i].mortonCode = int(keys[i])
    s, _, _ = oracle_scene_from_ctx(O, ctx, sc.cam, sc.params, svp, sc.ext)
    ref = O.gather_render(O.beam_scene(s, sorted_beams, data, nodes, n, 0, 0, 0.9), fr)
    assert_bitexact(gpu, ref, f"gather over {n} beams in a chain")
    assert gpu[..., 0].max() > 0.0
