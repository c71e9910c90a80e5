"""The one-workgroup generator's exact selection where errors tie: buckets of tied nodes
below, at and above the size that is ranked directly, in one to three dims; regions,
errors and bins bit for bit those of the parallel rounds (VMX_DEFER=0)."""
import numpy as np
import pytest

import viltrum_amd as V
from viltrum_amd import integrands as I

pytestmark = pytest.mark.gpu

FLAT = {d: I.poly([(0.7, (0,) * d)], d) for d in (1, 2, 3)}  # every region of a size ties
# flat but for a corner: distinct errors beside tied ones
CORNER = {d: I.poly([(0.7, (0,) * d)], d, step=([1.0] * d, 0.9 * d, 0.5)) for d in (1, 2, 3)}


# a level of a flat tree holds 2^k tied nodes: budgets inside levels of 64 to 1024 nodes,
# one node into a level, all but one node of it, and at its end
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("n", [65, 100, 255, 256, 257, 258, 300, 511, 513, 900, 1024, 1600, 2047])
@pytest.mark.parametrize("f", [*FLAT.values(), *CORNER.values()], ids=["flat1", "flat2", "flat3", "corner1", "corner2",
                                                                       "corner3"])
def test_ties(ctx, monkeypatch, f, n, dt):
    res = {1: (30,), 2: (9, 8), 3: (7, 5)}[f.dim]
    out = []
    for rounds in (True, False):
        if rounds:
            monkeypatch.setenv("VMX_DEFER", "0")
        else:
            monkeypatch.delenv("VMX_DEFER")
        it = V.Integrator(n - 1, 2, 4)
        b = np.zeros(res, dtype=dt)
        V.integrate(it, b, f, V.range_primary(f.dim), ctx=ctx)
        out.append((b, ctx.export_regions(f.dim), it.last_stats.ties_unresolved))
    (b0, r0, t0), (b1, r1, t1) = out
    for key in ("lo", "hi", "nodes", "err", "dim"):
        assert np.array_equal(r0[key], r1[key]), key
    assert np.array_equal(b0, b1) and t0 == t1
