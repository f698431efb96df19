"""Grid uploads whose rows and columns cross the conversion's 32 x 32 tiles, and
skip-grid distances along each axis beyond and within their limit of 16."""
import numpy as np
import pytest

from gpu_util import assert_bitexact

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(1, 1, 1), (33, 2, 31), (70, 3, 45), (32, 5, 64)])
@pytest.mark.parametrize("src,storage", [(np.float32, 0), (np.float32, 1), (np.float16, 0), (np.float16, 1)])
@pytest.mark.parametrize("layout", [0, 1])
def test_z_fastest_upload(ctx, S, dims, src, storage, layout):
    nx, ny, nz = dims
    g = np.random.default_rng(nx).random((nx, ny, nz)).astype(src)   # z fastest
    ctx.set_grid_layout(layout)
    ctx.upload_grid(g, 0.01, layout=S.CR_LAYOUT_Z_FASTEST, storage=storage)
    want = g.transpose(2, 1, 0).astype(np.float16 if storage else np.float32).astype(np.float32)
    assert_bitexact(ctx.download_grid(), np.ascontiguousarray(want), f"{dims}, {src.__name__} to {storage}")


@pytest.mark.parametrize("dims", [(88, 4, 4), (4, 88, 4), (4, 4, 88), (40, 24, 76)])
@pytest.mark.parametrize("occupied", [[], [0], [-1], [0, -1], [7]])
def test_skip_distances(ctx, cfg, S, dims, occupied):
    nx, ny, nz = dims
    ctx.set_render_ext(cfg.render_ext(majorant_brick=4))
    g = np.zeros((nz, ny, nx), np.float32)
    for o in occupied:
        g.reshape(-1)[o if o != 7 else g.size // 2 + nx // 3] = 0.5
    ctx.upload_grid(g, 0.01)
    maj, skip = ctx.majorants(), ctx.skip_grid()
    occ = np.argwhere(maj > 0)
    cl = ctx.cloud()
    want = (maj * np.float32(cl.densityScaling) / np.float32(cl.baseScaling)).astype(np.float32)
    for idx in np.argwhere(maj == 0):
        want[tuple(idx)] = -float(16 if len(occ) == 0 else min(16, int(np.abs(occ - idx).max(axis=1).min())))
    assert_bitexact(skip, want, f"{dims}, occupied {occupied}")
