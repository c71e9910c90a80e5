"""Which way a call's regions were generated, as vmx_last_generation reports it: one
workgroup per integral, parallel rounds, or the one after the other."""
import numpy as np
import pytest

import viltrum_amd as V
from viltrum_amd import hip
from viltrum_amd import integrands as I

pytestmark = pytest.mark.gpu

BLOBS = I.config4_integrand(11)


def _integrate(ctx, f, n, res=(24, 17), dt=np.float32, **kw):
    it = V.Integrator(n - 1, 2, 3, **kw)
    V.integrate(it, np.zeros(res, dtype=dt), f, V.range_primary(f.dim), ctx=ctx)
    g = ctx.last_generation()
    assert it.last_stats.rounds == g["workgroup_steps"] + g["rounds"]
    return g


def _ways(g):
    return g["workgroup_steps"] > 0, g["rounds"] > 0, g["handovers"]


def test_ways_are_told_apart(ctx, monkeypatch):
    assert _ways(_integrate(ctx, BLOBS, 600)) == (True, False, 0)
    assert _ways(_integrate(ctx, BLOBS, 20000)) == (True, True, 0)  # alone: starts in a workgroup
    assert _ways(_integrate(ctx, I.config5(2), 300)) == (False, True, 0)  # 5 dims
    monkeypatch.setenv("VMX_DEFER", "0")
    assert _ways(_integrate(ctx, BLOBS, 600)) == (False, True, 0)


def test_groups_of_a_batch_are_summed_and_given_regions_have_none(ctx):
    fs = [BLOBS, I.config5(2)]
    bufs = [hip.DeviceBuffer(16 * 16 * 4) for _ in fs]
    ps = [V.Integrator(299, 2, 3).problem(f, (16, 16), V.range_primary(f.dim), V.F32) for f in fs]
    ctx.integrate_batch(ps, fs, [b.address for b in bufs])
    assert _ways(ctx.last_generation()) == (True, True, 0)
    for b in bufs:
        b.free()
    it = V.Integrator(299, 2, 3)
    b = np.zeros((16, 16), dtype=np.float32)
    V.integrate(it, b, BLOBS, V.range_primary(2), ctx=ctx)
    V.integrate_regions(it, b, BLOBS, V.range_primary(2), ctx.export_regions(2), ctx=ctx)
    assert _ways(ctx.last_generation()) == (False, False, 0)


POLY3 = I.poly([(1.0, (1, 2, 0)), (0.5, (2, 0, 1)), (0.3, (3, 1, 2))], 3, step=([1, 1, 1], 1.5, 0.25))
LONG3 = I.poly([(0.1 * (k + 1), (k % 4, (k + 1) % 4, (k + 2) % 3)) for k in range(12)], 3)
MOVING8 = I.moving_blobs(3, 8)


# both sides of the choice, at sizes where one generator was measured 10 % or more ahead
@pytest.mark.parametrize("f,dt,jobs,n,workgroup", [
    (POLY3, np.float64, 1, 1600, False), (MOVING8, np.float64, 1, 800, False), (POLY3, np.float32, 1, 4000, False),
    (LONG3, np.float32, 1, 2400, False), (MOVING8, np.float32, 1, 6000, False), (POLY3, np.float64, 1, 20, True),
    (MOVING8, np.float32, 1, 800, True), (BLOBS, np.float32, 1, 6144, True), (BLOBS, np.float64, 1, 4000, True),
    (POLY3, np.float64, 64, 400, True), (POLY3, np.float32, 64, 2400, True)],
    ids=lambda v: getattr(v, "__name__", str(v)) if not hasattr(v, "desc") else "f%d" % v.dim)
def test_the_faster_generator_is_chosen(ctx, f, dt, jobs, n, workgroup):
    res = (24, 17)
    ps = [V.Integrator(n - 1, 1, i).problem(f, res, V.range_primary(f.dim), V.F32 if dt == np.float32 else V.F64)
          for i in range(jobs)]
    bufs = [hip.DeviceBuffer(24 * 17 * 8) for _ in ps]
    ctx.integrate_batch(ps, [f] * jobs, [b.address for b in bufs])
    for b in bufs:
        b.free()
    g = ctx.last_generation()
    assert (g["rounds"] == 0) == workgroup and g["handovers"] == 0, g


def test_starts_in_a_workgroup_where_that_gains(ctx):
    assert _ways(_integrate(ctx, MOVING8, 20000)) == (True, True, 0)
    assert _ways(_integrate(ctx, POLY3, 20000, dt=np.float64)) == (False, True, 0)


# the series of a wave's 64 samples run to the longest: 81 terms on average at decay 0.95,
# where 1600 regions of 3 dims take 2345 us in a workgroup, 1093 by rounds
@pytest.mark.parametrize("rd,decay,mc,n,workgroup", [(3, 0.95, 1, 1600, False), (3, 0.75, 1, 1600, False),
                                                     (2, 0.95, 1, 1600, False), (2, 0.75, 1, 400, True),
                                                     (1, 0.3, 4, 1600, True)])
def test_series_over_an_infinite_range(ctx, rd, decay, mc, n, workgroup):
    it = V.integrator_crespo2021_infinite(rd, n - 1, mc, 2, seed=3)
    V.integrate(it, np.zeros((9, 8, 7)[:rd], dtype=np.float32), I.dyson(decay), V.range_primary_infinite(), ctx=ctx)
    assert (ctx.last_generation()["rounds"] == 0) == workgroup


def test_generation_time_of_small_integrals(ctx):
    """8 times the regions take several times the steps: the time is the generation's, not its
    launch's, and the phases do not count it twice."""
    ms = {}
    for n in (700, 6000):
        it = V.Integrator(n - 1, 2, 3)
        best = 1e9
        for _ in range(8):
            b = np.zeros((24, 17), dtype=np.float32)
            V.integrate(it, b, BLOBS, V.range_primary(2), ctx=ctx)
            s = it.last_stats
            assert ctx.last_generation()["rounds"] == 0
            assert s.ms_generate + s.ms_select + s.ms_stratify <= s.ms_total and s.ms_stratify >= 0
            best = min(best, s.ms_generate)
        ms[n] = best
    assert ms[6000] > 1.5 * ms[700] > 0.05, ms
