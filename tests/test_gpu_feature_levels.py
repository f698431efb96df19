"""The stencil features where the levels staged in LDS begin: chains of levels that
just fit into it (38^3 from level 1 on, 1000 x 2 x 2 from level 0 on) and just do
not (40^3), and the sizes around them."""
import pytest

from test_gpu_features import test_features_bitexact as check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(38, 38, 38), (39, 38, 38), (40, 40, 40), (76, 75, 74), (144, 130, 129), (1000, 2, 2),
                                      (8192, 1, 1), (8191, 1, 1), (2, 2, 2)])
def test_staged_levels(ctx, cfg, S, nx, ny, nz):
    check(ctx, cfg, S, nx, ny, nz, 1.0)
