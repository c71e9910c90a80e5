"""Integrals that one workgroup cannot finish (its pool full of tied errors, its share of
the tree used up) go to the parallel rounds, which generate them or refuse them: regions
and bins bit for bit those of the rounds alone (VMX_DEFER=0), and nothing that later calls
of the class depend on is changed by it."""
import numpy as np
import pytest

import viltrum_amd as V
from viltrum_amd import hip
from viltrum_amd import integrands as I

pytestmark = pytest.mark.gpu

CONST = I.poly([(0.7, (0, 0))], 2)  # every region of a size ties
POLY2 = I.poly([(1.0, (1, 2)), (0.5, (3, 0)), (0.25, (0, 0))], 2, step=([1, 1], 1.1, 0.5))


@pytest.fixture
def fresh():
    c = V.Context(0)
    yield c
    c.close()


def _noalloc(ctx, f, integ, res):
    buf = hip.DeviceBuffer(4 * int(np.prod(res)))
    try:
        buf.zero()
        ctx.integrate_device_noalloc(integ.problem(f, res, V.range_primary(2), V.F32), f, buf.address)
        return buf.to_host(np.zeros(res, dtype=np.float32))
    finally:
        buf.free()


def _bins(ctx, f, integ, res, dt=np.float32):
    b = np.zeros(res, dtype=dt)
    V.integrate(integ, b, f, V.range_primary(f.dim), ctx=ctx)
    return b


def test_a_refused_call_leaves_later_calls_their_memory(fresh):
    """Every FP32 error of a constant is 0 under the absolute heuristic, so no threshold
    ends the refinement and the call is refused whatever its budget.  16384 regions at 64
    nodes each would not fit the no-alloc scratch; at 8 they do."""
    res, small, large = (512, 512), V.Integrator(19, 2, 3, heuristic=V.HEUR_DEFAULT_ABSOLUTE), V.Integrator(16383, 2, 3)
    want = _noalloc(fresh, POLY2, large, res)
    with pytest.raises(V.VmxError, match="node capacity"):
        _bins(fresh, CONST, small, res)
    assert np.array_equal(_noalloc(fresh, POLY2, large, res), want)
    assert np.array_equal(_bins(fresh, POLY2, large, res), want)


@pytest.mark.parametrize("n", [4500, 6144])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_a_full_pool_is_generated_by_rounds(fresh, monkeypatch, n, dt):
    integ = V.Integrator(n - 1, 2, 5)
    got = _bins(fresh, CONST, integ, (40, 24), dt)
    regions = fresh.export_regions(2)
    g = fresh.last_generation()
    assert g["handovers"] == 1 and g["workgroup_steps"] > 0 and g["rounds"] > 0
    monkeypatch.setenv("VMX_DEFER", "0")
    assert np.array_equal(_bins(fresh, CONST, integ, (40, 24), dt), got)
    assert fresh.last_generation()["handovers"] == 0
    for k, v in fresh.export_regions(2).items():
        assert np.array_equal(v, regions[k]), k


def test_a_full_pool_in_a_batch_and_without_allocation(fresh, monkeypatch):
    integ = V.Integrator(4499, 2, 5)
    got = _noalloc(fresh, CONST, integ, (40, 24))
    assert fresh.last_generation()["handovers"] == 1
    assert np.array_equal(_bins(fresh, CONST, integ, (40, 24)), got)
    fs, its = [POLY2, CONST, POLY2], [V.Integrator(n - 1, 2, 7 + n) for n in (300, 4500, 1200)]
    out = []
    ctx = V.Context(0)
    try:
        for rounds in (False, True):
            if rounds:
                monkeypatch.setenv("VMX_DEFER", "0")
            bufs = [hip.DeviceBuffer(4 * 40 * 24) for _ in fs]
            ctx.integrate_batch([it.problem(f, (40, 24), V.range_primary(2), V.F32) for f, it in zip(fs, its)], fs,
                                [b.address for b in bufs])
            assert ctx.last_generation()["handovers"] == (0 if rounds else 1)
            out.append([b.to_host(np.zeros((40, 24), dtype=np.float32)) for b in bufs])
            for b in bufs:
                b.free()
    finally:
        ctx.close()
    for x, y in zip(*out):
        assert np.array_equal(x, y)


def test_one_handover_does_not_set_the_class(fresh):
    """After a handover the next call of the class runs the rounds and the one after it
    tries the workgroup again; while they keep failing the tries thin out."""
    tied, plain = V.Integrator(4499, 2, 5), V.Integrator(4499, 2, 6)
    _bins(fresh, CONST, tied, (40, 24))
    assert fresh.last_generation()["handovers"] == 1
    seen = []
    for _ in range(3):
        _bins(fresh, POLY2, plain, (40, 24))
        g = fresh.last_generation()
        assert g["handovers"] == 0
        seen.append(g["rounds"] == 0)
    assert seen == [False, True, True]
    tries = 0
    for _ in range(100):
        _bins(fresh, CONST, tied, (40, 24))
        tries += fresh.last_generation()["handovers"]
    assert tries == 6  # at calls 1, 3, 7, 15, 31 and 63


# FP64 trees of 3 dims have the smallest pool, 1536 nodes
@pytest.mark.parametrize("deepen", ["0", "1"])
@pytest.mark.parametrize("n", [2000, 2047, 2048, 2049, 2560, 2561, 3000, 3073, 4000, 6144])
def test_no_handover_by_size_alone(fresh, monkeypatch, n, deepen):
    monkeypatch.setenv("VMX_DEEPEN", deepen)
    f = I.poly([(1.0, (1, 2, 0)), (0.5, (2, 0, 1)), (0.3, (3, 1, 2))], 3, step=([1, 1, 1], 1.5, 0.25))
    ps = [V.Integrator(n - 1, 1, i).problem(f, (6, 5), V.range_primary(3), V.F64) for i in range(64)]
    bufs = [hip.DeviceBuffer(6 * 5 * 8) for _ in ps]
    fresh.integrate_batch(ps, [f] * len(ps), [b.address for b in bufs])
    for b in bufs:
        b.free()
    assert fresh.last_generation()["handovers"] == 0


def test_more_room_in_the_tree(fresh, monkeypatch):
    """A constant in 3 dims: 100 regions take 1023 nodes, more than 8 a region and 64.  The
    rounds find the room, the class keeps it, and the workgroup has it from then on."""
    f, integ = I.poly([(0.7, (0, 0, 0))], 3), V.Integrator(99, 2, 5)
    ways, outs = [], []
    for k in range(4):
        if k == 3:
            monkeypatch.setenv("VMX_DEFER", "0")
        outs.append((_bins(fresh, f, integ, (7, 5)), fresh.export_regions(3)))
        g = fresh.last_generation()
        ways.append((g["workgroup_steps"] > 0, g["rounds"] > 0, g["handovers"]))
    assert ways == [(True, True, 1), (False, True, 0), (True, False, 0), (False, True, 0)]
    for b, r in outs[1:]:
        assert np.array_equal(b, outs[0][0])
        for key, v in r.items():
            assert np.array_equal(v, outs[0][1][key]), key


# one integral that starts in a workgroup and goes on in the deferred rounds (65536 regions
# and more), with the candidates' counts and the histogram that the workgroup left
@pytest.mark.parametrize("f,res,dt", [(POLY2, (24, 20), np.float32), (POLY2, (24, 20), np.float64),
                                      (I.config4_integrand(3), (40, 30), np.float32),
                                      (I.moving_blobs(3, 6), (16, 12), np.float32),
                                      (I.poly([(1.0, (3,)), (0.5, (1,))], 1, step=([1.0], 0.37, 0.25)), (40,), np.float32)],
                         ids=["poly2", "poly2_f64", "blobs2", "moving3", "poly1"])
def test_goes_on_in_deferred_rounds(fresh, monkeypatch, f, res, dt):
    integ = V.Integrator(69999, 1, 5)
    got = _bins(fresh, f, integ, res, dt), fresh.export_regions(f.dim)
    g = fresh.last_generation()
    assert g["workgroup_steps"] > 0 and g["rounds"] > 0 and g["handovers"] == 0
    monkeypatch.setenv("VMX_DEFER", "0")
    want = _bins(fresh, f, integ, res, dt), fresh.export_regions(f.dim)
    assert fresh.last_generation()["workgroup_steps"] == 0
    assert np.array_equal(got[0], want[0])
    for key, v in want[1].items():
        assert np.array_equal(v, got[1][key]), key


@pytest.mark.parametrize("n", [6145, 8192, 20000, 70000])
@pytest.mark.parametrize("f,res", [(I.config4_integrand(3), (32, 20)), (I.poly([(1.0, (3,)), (0.5, (1,))], 1), (32,))],
                         ids=["blobs2", "poly1"])
def test_goes_on_in_learned_rounds(fresh, monkeypatch, f, res, n):
    p = (np.random.default_rng(5).standard_normal(V.refiner_size(f.dim)[0]) * 0.1).astype(np.float32)
    p[-2], p[-1] = -20.0, 4.0  # mu, sigma
    fresh.refiner_set(f.dim, p)
    integ = V.Integrator(n - 1, 1, 5, refiner=V.REFINER_LEARNED)
    got = _bins(fresh, f, integ, res), fresh.export_regions(f.dim)
    g = fresh.last_generation()
    assert g["workgroup_steps"] > 0 and g["rounds"] > 0 and g["handovers"] == 0
    monkeypatch.setenv("VMX_DEFER", "0")
    want = _bins(fresh, f, integ, res), fresh.export_regions(f.dim)
    assert np.array_equal(got[0], want[0])
    for key, v in want[1].items():
        assert np.array_equal(v, got[1][key]), key
