"""A theta block's sorting of its own candidates (deferred rounds, integrals of up to 32768
regions) keeps the regions of the undeferred rounds, with 1 to many times the 4096
candidates of one pass, and with none."""
import numpy as np
import pytest

import viltrum_amd as V
from viltrum_amd import hip
from viltrum_amd import integrands as I

pytestmark = pytest.mark.gpu

CONST = I.poly([(0.7, (0, 0))], 2)  # every region of a size ties: a round's candidates all split or all wait


def _deferred_equals_undeferred(ctx, monkeypatch, scalar, dt, k, its):
    fs = [CONST if n == 20000 else I.c1_family(20 + i, 8) for i, n in enumerate(its)]
    ps = [V.Integrator(n, 2, 30 + i).problem(f, (24, 24), V.range_primary(2), scalar)
          for i, (f, n) in enumerate(zip(fs, its))]
    outs = []
    for d in (0, k):
        monkeypatch.setenv("VMX_DEFER", str(d))
        bufs = [hip.DeviceBuffer(24 * 24 * np.dtype(dt).itemsize) for _ in ps]
        ctx.integrate_batch(ps, fs, [b.address for b in bufs])
        outs.append([b.to_host(np.zeros((24, 24), dtype=dt)) for b in bufs])
        for b in bufs:
            b.free()
    for i, (x, y) in enumerate(zip(*outs)):
        assert np.array_equal(x, y), its[i]


@pytest.mark.parametrize("scalar,dt", [(V.F32, np.float32), (V.F64, np.float64)])
@pytest.mark.parametrize("k", [1, 2, 64])
def test_candidates_sorted_by_theta_blocks(ctx, monkeypatch, scalar, dt, k):
    _deferred_equals_undeferred(ctx, monkeypatch, scalar, dt, k, [0, 1, 1023, 4096, 9000, 32767, 20000])


# one integral above 32768 regions sends the batch's candidates through the grid: runs that
# hold several integrals, end inside one, and integrals without candidates between others
@pytest.mark.parametrize("scalar,dt", [(V.F32, np.float32), (V.F64, np.float64)])
@pytest.mark.parametrize("k", [1, 64])
def test_candidates_sorted_by_the_grid(ctx, monkeypatch, scalar, dt, k):
    _deferred_equals_undeferred(ctx, monkeypatch, scalar, dt, k, [0, 300, 0, 0, 5, 1023, 40000, 0, 20000, 4096, 0])
