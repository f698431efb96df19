"""The one-workgroup sort of small beam sets (at most 8192): sizes around the
waves' groups of 128, powers of two and its limit, with many equal keys,
against a stable sort."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_ppb import random_beams, setup_c1

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 63, 64, 65, 127, 128, 129, 257, 1023, 2048, 4095, 4096, 4097, 8191, 8192, 8193])
@pytest.mark.parametrize("dup", [0.0, 0.7])
def test_small_sort_is_stable(ctx, cfg, S, O, n, dup):
    sc, cloud, _ = setup_c1(ctx, cfg, S, size=16)
    beams, data = random_beams(S, n, seed=n, dup_frac=dup)
    ctx.upload_beams(beams, data)
    ctx.lbvh_build()
    keys, perm, _ = ctx.lbvh_download()
    codes = np.empty(n, np.uint32)
    O.lib.or_beam_morton30(beams, n, (C.c_float * 3)(*cloud.bounds[0][:3]), (C.c_float * 3)(*cloud.bounds[1][:3]),
                           codes.ctypes.data)
    want = np.argsort(codes, kind="stable")
    np.testing.assert_array_equal(perm, want)
    np.testing.assert_array_equal(keys, codes[want])
