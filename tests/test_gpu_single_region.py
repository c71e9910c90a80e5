"""The per-bin kernel's loop for waves of single-region bins, and its tiles of 16 x 16 bins.
In a batch with a roulette integral every integral runs the general loop (region draw and
list per sample), on the same words and with the same arithmetic: bins equal bit for bit."""
import numpy as np
import pytest

import viltrum_amd as V
from viltrum_amd import hip
from viltrum_amd import integrands as I

pytestmark = pytest.mark.gpu

P1 = I.poly([(1.0, (3,)), (0.5, (1,))], 1, step=([1.0], 0.37, 0.25))
S2 = I.poly([(1.0, (1, 2)), (0.5, (3, 0)), (0.25, (0, 0))], 2, step=([1, 1], 1.1, 0.5))


def _general(ctx, integ, f, res):
    """The integral's bins from a batch that holds a roulette integral too."""
    rr = V.integrator_variance_reduction_rr_integral(6, 2, 9)
    small = (4,) * len(res)
    items = [(integ, res), (rr, small)]
    bufs = [hip.DeviceBuffer(int(np.prod(r)) * 4) for _, r in items]
    for b in bufs:
        b.zero()  # CV_ALPHA1 adds to its bins
    ctx.integrate_batch([i.problem(f, r, V.range_primary(f.dim), V.F32) for i, r in items], [f, f],
                        [b.address for b in bufs])
    out = bufs[0].to_host(np.zeros(res, dtype=np.float32))
    for b in bufs:
        b.free()
    return out


# grids at the edges of the tiles (one, two, partial, narrow: runs of 256 bins); budgets from
# one region over all bins to several per bin; sample counts below, at and beyond a group of 4
@pytest.mark.parametrize("f,res", [
    (P1, (15,)), (P1, (300,)), (S2, (15, 16)), (S2, (16, 15)), (S2, (16, 16)), (S2, (17, 33)), (S2, (31, 16)),
    (S2, (16, 1000)), (I.config1(), (64, 48)), (I.c1_family(5, 30), (100, 37))], ids=lambda v: getattr(v, "name", str(v)))
def test_single_region_bins(ctx, f, res):
    for it, spp, form in [(0, 5, V.FORM_VR_OPTIMIZE), (40, 1, V.FORM_VR_OPTIMIZE), (40, 3, V.FORM_VR_FIXED),
                          (40, 16, V.FORM_CV_ALPHA1), (900, 4, V.FORM_VR_OPTIMIZE), (900, 18, V.FORM_VR_FIXED),
                          (40, 0, V.FORM_VR_OPTIMIZE)]:
        integ = V.Integrator(it, spp, 3, form=form, alpha=0.7)
        b = np.zeros(res, dtype=np.float32)
        V.integrate(integ, b, f, V.range_primary(f.dim), ctx=ctx)
        assert np.array_equal(b, _general(ctx, integ, f, res)), (it, spp, form)
