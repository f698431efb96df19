"""The stencil features bit for bit against the same float32 operations in
NumPy: box extents that divide by multiplication (powers of two), by residuals
(others) and by IEEE division (extents out of range), levels in LDS and in
memory, one-voxel axes, and points on the faces, at the corners and outside."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

F = np.float32


def mips(grid):
    """Levels 0..7, indexed [z, y, x]: means of the existing voxels of 2x2x2 blocks, added x first."""
    out = [grid]
    for _ in range(7):
        g = out[-1]
        d = [(s + 1) // 2 for s in g.shape]
        acc, cnt = np.zeros(d, F), np.zeros(d, F)
        for c in range(8):
            part = g[(c >> 2)::2, ((c >> 1) & 1)::2, (c & 1)::2]
            sl = tuple(slice(0, s) for s in part.shape)
            acc[sl] = acc[sl] + part
            cnt[sl] += F(1)
        out.append(acc / cnt)
    return out


def trilinear(g, n):
    def axis(n, N):
        u = np.minimum(np.maximum(n * F(N) - F(0.5), F(-1)), F(N))
        fl = np.floor(u)
        i = fl.astype(np.int64)
        return np.clip(i, 0, N - 1), np.clip(i + 1, 0, N - 1), u - fl
    nz, ny, nx = g.shape
    (x0, x1, a), (y0, y1, b), (z0, z1, c) = axis(n[:, 0], nx), axis(n[:, 1], ny), axis(n[:, 2], nz)
    oa, ob, oc = F(1) - a, F(1) - b, F(1) - c
    c00 = g[z0, y0, x0] * oa + g[z0, y0, x1] * a
    c10 = g[z0, y1, x0] * oa + g[z0, y1, x1] * a
    c01 = g[z1, y0, x0] * oa + g[z1, y0, x1] * a
    c11 = g[z1, y1, x0] * oa + g[z1, y1, x1] * a
    return (c00 * ob + c10 * b) * oc + (c01 * ob + c11 * b) * c


def bf16(v):
    u = v.astype(F).view(np.uint32).astype(np.uint64)
    return ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)


def features(levels, b0, b1, sscale, h0, x, w, light):
    ez = [F(-light[k]) for k in range(3)]
    sz = F(1) if ez[2] >= 0 else F(-1)
    aa = ez[1] / (F(1) + np.abs(ez[2]))
    bb, cc = ez[1] * aa, -ez[0] * aa
    ex = [ez[2] + sz * bb, sz * cc, -ez[0]]
    ey = [cc, F(1) - bb, -sz * ez[1]]
    out = np.zeros((len(x), 224), np.uint16)
    h, j = F(h0), 0
    for g in levels:
        for t in range(27):
            fi, fj, fl = F(t % 3 - 1) * h, F(t // 3 % 3 - 1) * h, F(t // 9 - 1) * h
            p = np.stack([x[:, k] + ((fi * ex[k] + fj * ey[k]) + fl * ez[k]) for k in range(3)], axis=1)
            inside = np.all(p >= b0, axis=1) & np.all(p <= b1, axis=1)
            d = np.where(inside, trilinear(g, (p - b0) / (b1 - b0)), F(0))
            out[:, j] = bf16((d * sscale) * h)
            j += 1
        h = h * F(2)
    c = (w[:, 0] * ez[0] + w[:, 1] * ez[1]) + w[:, 2] * ez[2]
    out[:, 216], out[:, 217] = bf16(c), bf16(c * c)
    return out


@pytest.mark.parametrize("nx,ny,nz,scale", [(36, 36, 36, 1.0), (64, 32, 16, 1.0), (1, 9, 5, 3.7), (150, 7, 41, 1.0),
                                            (21, 30, 17, 1e21)])
def test_features_bitexact(ctx, cfg, S, nx, ny, nz, scale):
    rng = np.random.default_rng(nx)
    grid = (rng.random((nz, ny, nx)) ** 3).astype(F)
    sc = cfg.c1(width=16, height=16, size=16, sv_axis=16)
    cloud, svp = sc.setup(ctx, build_sv=False)
    ctx.upload_grid(grid, 1.0 / max(nx, ny, nz))
    cloud = ctx.cloud()
    for k in range(3):
        cloud.bounds[0][k] *= scale
        cloud.bounds[1][k] *= scale
    ctx.set_cloud(cloud)
    ctx.learn_build_mips()
    b0, b1 = np.array(cloud.bounds[0][:3], F), np.array(cloud.bounds[1][:3], F)
    n = 700   # two whole workgroups and part of a third
    x = (b0 + (b1 - b0) * rng.uniform(-0.1, 1.1, (n, 3)).astype(F)).astype(F)
    for i in range(27):   # corners, edges, faces and the centre
        x[i] = [(b0[k], b1[k], (b0[k] + b1[k]) / F(2))[(i // 3 ** k) % 3] for k in range(3)]
    w = rng.standard_normal((n, 3)).astype(F)
    pts = np.zeros((n, 8), F)
    pts[:, :3], pts[:, 3:6] = x, w
    X = np.empty((n, 224), np.uint16)
    ctx.check(ctx.lib.cr_learn_features(ctx.h, pts.ctypes.data, n, X.ctypes.data), "features")
    light = np.array(svp.lightDirection[:3], F)
    h0 = (b1[0] - b0[0]) / F(nx)
    with np.errstate(all="ignore"):
        ref = features(mips(grid), b0, b1, F(cloud.densityScaling) / F(cloud.baseScaling), h0, x, w, light)
    bad = np.argwhere(X != ref)
    assert len(bad) == 0, f"{len(bad)} of {X.size} differ; first {bad[0]}: {X[tuple(bad[0])]:#x} {ref[tuple(bad[0])]:#x}"
