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
