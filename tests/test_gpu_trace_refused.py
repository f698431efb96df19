"""Traces of more than 2^28 photon deposits or beam data records are refused, and
give their records' memory back."""
import ctypes as C

import pytest

from test_gpu_ppm import setup as ppm_setup

pytestmark = pytest.mark.gpu


@pytest.fixture()
def own(pkg):
    c = pkg.Context(0)
    yield c
    c.close()


def free_bytes():
    f, t = C.c_size_t(), C.c_size_t()
    assert C.CDLL("libamdhip64.so.7").hipMemGetInfo(C.byref(f), C.byref(t)) == 0
    return f.value


def test_too_many_deposits(own, cfg, S, pkg):
    sc, cloud, svp, pm, p = ppm_setup(own, cfg, S, pkg)
    cloud.densityScaling *= 30.0
    own.set_cloud(cloud)
    pm.absorption = 0.0
    own.set_photon_map(pm)
    p.numPaths = 1 << 24
    own.synchronize()
    before = free_bytes()
    n = C.c_uint32()
    assert own.lib.cr_ppm_trace(own.h, 3, C.byref(p), C.byref(n)) == S.CR_ERR_CAPACITY
    assert before - free_bytes() < 2 << 30
    p.numPaths = 1000
    assert own.ppm_trace(3, p) > 1000


def test_too_many_beam_data(own, cfg, S):
    sc = cfg.c1(width=16, height=16, size=32, sv_axis=16)
    sc.setup(own, build_sv=False)
    # one segment of beam per record: the path that fills max_beams goes on past it
    p = cfg.beam_params(1 << 26, seed=5, radius=2.0, albedo=1.0, max_interactions=64)
    own.synchronize()
    before = free_bytes()
    n, d = C.c_uint32(), C.c_uint32()
    assert own.lib.cr_ppb_trace_beams(own.h, C.byref(p), 1 << 28, C.byref(n), C.byref(d)) == S.CR_ERR_CAPACITY
    assert before - free_bytes() < 2 << 30
    p.numPaths = 1000
    assert own.trace_beams(p, 1 << 20)[1] > 1000
