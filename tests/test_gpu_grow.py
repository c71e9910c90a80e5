"""One workgroup generating an integral's regions (csrc/grow.h) gives exactly the regions of
the round kernels: boxes, node values, errors, split dims and bins bit for bit.  VMX_DEFER=0
sends a call through the undeferred rounds."""
import numpy as np
import pytest

import viltrum_amd as V
from viltrum_amd import hip
from viltrum_amd import integrands as I
from viltrum_amd import refiner as R

pytestmark = pytest.mark.gpu

POLY1 = I.poly([(1.0, (3,)), (0.5, (1,))], 1, step=([1.0], 0.37, 0.25))
POLY3 = I.poly([(1.0, (1, 2, 0)), (0.5, (2, 0, 1)), (0.3, (3, 1, 2))], 3, step=([1, 1, 1], 1.5, 0.25))
CONST = I.poly([(0.7, (0, 0))], 2)  # every region of a size ties
EVEN = I.poly([(1.0, (4, 0)), (1.0, (0, 4))], 2)  # symmetric: ties between dims and regions


def _both(ctx, monkeypatch, f, res, integ, dt):
    out = []
    for rounds in (True, False):
        if rounds:
            monkeypatch.setenv("VMX_DEFER", "0")
        else:
            monkeypatch.delenv("VMX_DEFER")
        b = np.zeros(res, dtype=dt)
        V.integrate(integ, b, f, V.range_primary(f.dim), ctx=ctx)
        out.append((b, ctx.export_regions(f.dim)))
    (b0, r0), (b1, r1) = out
    for key in ("lo", "hi", "nodes", "err", "dim"):
        assert np.array_equal(r0[key], r1[key]), key
    assert np.array_equal(b0, b1)


# budgets around the edges of a step (128 and 256 splits), of a wave's run of positions in
# the sort (512) and of the largest integral one workgroup takes (6144); beyond it a single
# integral starts there and goes on in the rounds
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 2, 3, 129, 257, 512, 513, 1025, 4096, 6144, 6145, 20000])
def test_budgets_2d(ctx, monkeypatch, n, dt):
    _both(ctx, monkeypatch, I.config4_integrand(11), (24, 17), V.integrator_crespo2021(n - 1, 4, seed=1), dt)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("heur", [V.HEUR_SIZE_RELATIVE, V.HEUR_DEFAULT_ABSOLUTE])
@pytest.mark.parametrize("f,res,n", [(POLY1, (40,), 700), (POLY3, (9, 7), 900), (POLY3, (5, 4, 3), 40),
                                     (I.moving_blobs(3, 6), (16, 12), 1200), (CONST, (8, 8), 3000),
                                     (EVEN, (16, 16), 2500), (I.c1_family(5, 64), (12, 12), 300)],
                         ids=["poly1", "poly3", "poly3_bins3", "moving3", "constant", "symmetric", "blobs64"])
def test_families(ctx, monkeypatch, f, res, n, heur, dt):
    if f is CONST and heur == V.HEUR_DEFAULT_ABSOLUTE and dt == np.float32:
        # every error rounds to 0, so no threshold ends the refinement: refused, as by the rounds
        with pytest.raises(V.VmxError, match="node capacity"):
            V.integrate(V.Integrator(n - 1, 3, 2, heuristic=heur), np.zeros(res, dtype=dt), f, V.range_primary(2),
                        ctx=ctx)
        return
    _both(ctx, monkeypatch, f, res, V.Integrator(n - 1, 3, 2, heuristic=heur), dt)


def test_fubini(ctx, monkeypatch):
    it = V.integrator_crespo2021_infinite(2, 600, 2, 4, seed=3)
    f = I.moving_blobs(8, 5)
    g, rng = it.prepare(f, V.range_primary(3))
    _both(ctx, monkeypatch, g, (20, 20), V.Integrator(600, 4, 3), np.float32)


@pytest.fixture
def random_network():
    ctx = V.Context(0)
    rng = np.random.default_rng(5)
    for dim in (1, 2):
        p = (rng.standard_normal(V.refiner_size(dim)[0]) * 0.1).astype(np.float32)
        p[-2], p[-1] = -20.0, 4.0  # mu, sigma
        ctx.refiner_set(dim, p)
    yield ctx
    ctx.close()


@pytest.mark.parametrize("n", [2, 40, 300, 1024, 4096])
def test_learned(random_network, monkeypatch, n):
    it = V.Integrator(n - 1, 3, 4, refiner=V.REFINER_LEARNED)
    _both(random_network, monkeypatch, R.held_out(1)[0], (32, 20), it, np.float32)
    _both(random_network, monkeypatch, POLY1, (32,), it, np.float32)


def test_batch_of_uneven_budgets_and_priorities(random_network, monkeypatch):
    """Jobs of one launch end at different steps; learned and heuristic ones mixed."""
    ctx = random_network
    fs = R.held_out(9)
    ns = [1, 2, 77, 128, 500, 1500, 2048, 3000, 4096]
    its = [V.Integrator(n - 1, 4, 10 + i, refiner=V.REFINER_LEARNED if i % 2 else V.REFINER_HEURISTIC)
           for i, n in enumerate(ns)]
    ps = [it.problem(f, (19, 23), V.range_primary(2), V.F32) for it, f in zip(its, fs)]
    bufs = [hip.DeviceBuffer(19 * 23 * 4) for _ in ps]
    out = []
    for rounds in (True, False):
        if rounds:
            monkeypatch.setenv("VMX_DEFER", "0")
        else:
            monkeypatch.delenv("VMX_DEFER")
        ctx.integrate_batch(ps, fs, [b.address for b in bufs])
        out.append([b.to_host(np.zeros((19, 23), dtype=np.float32)) for b in bufs])
    for b in bufs:
        b.free()
    for k, (x, y) in enumerate(zip(*out)):
        assert np.array_equal(x, y), k
