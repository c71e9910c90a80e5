"""Importance sampling in the per-bin kernel's loop for waves of single-region bins, where
what a box's draws share is formed once: bins equal bit for bit to the general loop's, which
every integral of a batch with a roulette integral runs."""
import numpy as np
import pytest

import viltrum_amd as V
from viltrum_amd import hip
from viltrum_amd import integrands as I

pytestmark = pytest.mark.gpu

P1 = I.poly([(1.0, (3,)), (0.5, (1,))], 1, step=([1.0], 0.37, 0.25))
S2 = I.poly([(1.0, (1, 2)), (0.5, (3, 0)), (0.25, (0, 0))], 2, step=([1, 1], 1.1, 0.5))


def _general(ctx, integ, f, res):
    items = [(integ, res), (V.integrator_variance_reduction_rr_integral(6, 2, 9), (4,) * len(res))]
    bufs = [hip.DeviceBuffer(int(np.prod(r)) * 4) for _, r in items]
    ctx.integrate_batch([i.problem(f, r, V.range_primary(f.dim), V.F32) for i, r in items], [f, f],
                        [b.address for b in bufs])
    out = bufs[0].to_host(np.zeros(res, dtype=np.float32))
    for b in bufs:
        b.free()
    return out


# 5 to 40 regions over hundreds to thousands of bins: most waves hold bins of one region
# each, some cross regions; sample counts below, at and beyond a group of 4
@pytest.mark.parametrize("form", [V.FORM_VR_OPTIMIZE_IMPORTANCE, V.FORM_VR_FIXED_IMPORTANCE,
                                  V.FORM_VR_OPTIMIZE_SAMPLING_RR, V.FORM_VR_FIXED_SAMPLING_RR])
@pytest.mark.parametrize("f,res", [(P1, (300,)), (P1, (1025,)), (S2, (64, 48)), (S2, (17, 33)), (S2, (15, 200)),
                                   (I.config1(), (100, 37)), (I.c1_family(5, 30), (64, 64))],
                         ids=lambda v: getattr(v, "name", str(v)))
def test_importance_in_single_region_bins(ctx, f, res, form):
    for it, spp in [(0, 5), (4, 1), (4, 3), (12, 4), (12, 16), (40, 18)]:
        integ = V.Integrator(it, spp, 3, form=form, alpha=0.7)
        b = np.zeros(res, dtype=np.float32)
        V.integrate(integ, b, f, V.range_primary(f.dim), ctx=ctx)
        assert np.array_equal(b, _general(ctx, integ, f, res)), (it, spp)
