"""The beam producer's second pass with more records than it has waves for: the
beams of a trace cut short are the first of the whole one's, every beam's data is
written, and a trace of more than 2^26 records runs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BEAM, DATA = 12, 20   # words of a beam and of a beam's data


def words(array, per):
    return np.frombuffer(array, np.uint32).reshape(-1, per)


def thin_cloud(ctx, cfg):
    sc = cfg.c1(width=16, height=16, size=32, sv_axis=16)
    sc.density_scaling *= 0.03
    sc.setup(ctx, build_sv=False)


def test_more_records_than_waves(ctx, cfg, S):
    thin_cloud(ctx, cfg)
    p = cfg.beam_params(9 << 19, seed=11, radius=0.4, albedo=1.0, max_interactions=4)
    cut = 1 << 20
    assert ctx.trace_beams(p, cut)[0] == cut
    first = words(ctx.download_beams()[0], BEAM).copy()
    nb, nd = ctx.trace_beams(p, 1 << 26)
    assert nd > 1 << 22 and nb > nd
    beams, data = ctx.download_beams()
    beams, data = words(beams, BEAM), words(data, DATA)
    assert np.array_equal(beams[:cut], first)
    assert np.all(data[:, :4] == data[0, 0]), "power of some beam's data"
    assert np.all(data[:, 4:].view(np.float32) > 0.0), "transmittance distances of some beam's data"
    # path by path and interaction by interaction, each beam's first segment where the last one's end was
    assert np.all(np.diff(beams[:, 8].astype(np.int64)) >= 0) and beams[-1, 8] == nd - 1
    lead = np.flatnonzero(np.diff(beams[:, 8], prepend=np.uint32(0xffffffff)))
    assert np.all(beams[lead, 9] == 0)
    ctx.trace_beams(p, 64)


def test_two_to_the_26_records(pkg, cfg, S):
    ctx = pkg.Context(0)
    thin_cloud(ctx, cfg)
    p = cfg.beam_params(1 << 26, seed=5, radius=2.0, albedo=1.0, max_interactions=4)
    nb, nd = ctx.trace_beams(p, 1 << 28)     # one segment of beam per record
    assert nb == nd > 1 << 26
    beams, data = ctx.download_beams()
    ctx.close()
    assert np.array_equal(words(beams, BEAM)[:, 8], np.arange(nd, dtype=np.uint32))
    power = words(data, DATA)[:, 0]
    assert np.all(power == power[0]) and power[0] != 0
