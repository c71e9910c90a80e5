"""Per-bin footprint lists: the passes over (bin, footprint) pairs and the merged marginals.
FP64 bins of the control variate alone (spp = 0) against the oracle, whose per-region sums
they regroup: a bin adds at most a few hundred terms of one sign and size, so 1e-12 relative
is several hundred units in the last place."""
import numpy as np
import pytest

import oracle_lib as O
import viltrum_amd as V
from viltrum_amd import integrands as I

pytestmark = pytest.mark.gpu

P1 = I.poly([(1.0, (2,)), (0.5, (1,))], 1, step=([1.0], 0.4, 0.5))
P2 = I.poly([(1.0, (1, 2)), (0.5, (3, 0)), (0.25, (0, 0))], 2, step=([1, 1], 1.1, 0.5))
P3 = I.poly([(1.0, (1, 2, 0)), (0.5, (2, 0, 1)), (0.25, (0, 0, 2))], 3, step=([1, 1, 1], 1.5, 0.25))
T3 = I.poly([(1.0, (0, 0, 4)), (0.5, (0, 0, 1))], 3)  # varies along the integrated dim only: one footprint
P4 = I.poly([(1.0, (1, 0, 2, 1)), (0.5, (0, 2, 1, 0)), (0.25, (0, 0, 0, 3))], 4, step=([1, 1, 1, 1], 2.0, 0.5))


# pair totals at the edges of a wave's 64 pairs and of its run: one region over 1 .. 1025
# bins; then many footprints of a few bins; merged footprints with 1, 2 and 3 bin dims
@pytest.mark.parametrize("f,res,it", [
    *[(P1, (n,), 0) for n in (1, 63, 64, 65, 255, 256, 257, 511, 513, 1025)],
    (P2, (33, 31), 700), (P2, (3, 2), 700), (P2, (200, 1), 300), (P1, (700,), 500),
    (P3, (17, 9), 500), (P3, (5, 4, 3), 300), (P3, (40,), 400), (T3, (24, 11), 120),
    (P4, (9, 7), 300), (P4, (6,), 200), (P4, (3, 4, 5), 200)], ids=lambda v: getattr(v, "name", str(v)))
def test_control_variate_bins(ctx, f, res, it):
    bins = np.zeros(res)
    V.integrate(V.Integrator(it, 0, 0), bins, f, V.range_primary(f.dim), ctx=ctx)
    want, _ = O.integrate(f, res, it, 0, 0, scalar=8)
    np.testing.assert_allclose(bins, want.reshape(res), rtol=1e-12, atol=1e-12 * np.abs(want).max())
