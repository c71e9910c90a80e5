"""The importance sampler's root by Newton's method (viltrum_amd/csrc/importance.h on the
host) against the exact root in 64 bits, and its draws where there is no such root.

Lines have node values k / 16, so their coefficients are exact in float, and are kept where
the pdf is at least 1/32 over [0, 1] and no coefficient is below the sampler's own 1e-3
cut-offs.  The target is formed in float from two values of the cdf and the linear and
constant coefficients are rounded to float: at most 8 roundings of half an ulp of cdf(1),
over the smallest slope; twice that, and an ulp of the result."""
import ctypes as C
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), "native"))
import build as native_build  # noqa: E402

H = C.CDLL(native_build.build())
FP = C.POINTER(C.c_float)
H.vmh_imp_sample_line.restype = C.c_float
H.vmh_imp_sample_line.argtypes = [C.c_float, C.c_float, C.c_float, FP]


def _draw(s, t0, t1, p):
    p = np.ascontiguousarray(p, dtype=np.float32)
    return H.vmh_imp_sample_line(s, t0, t1, p.ctypes.data_as(FP))


@pytest.mark.parametrize("box", ["whole", "wide", "narrow", "at 0", "at 1"])
def test_root_against_64_bits(box):
    rng = np.random.default_rng(len(box))
    checked = 0
    while checked < 4000:
        q = rng.integers(1, 33, 3) / 16.0
        c0, c1, c2 = q[0], -3 * q[0] + 4 * q[1] - q[2], 2 * q[0] - 4 * q[1] + 2 * q[2]
        t = np.linspace(0, 1, 257)
        low = ((c2 * t + c1) * t + c0).min()
        if low < 1 / 32:
            continue
        cdf = lambda x: ((c2 / 3 * x + c1 / 2) * x + c0) * x  # noqa: E731
        a, b = np.sort(rng.random(2))
        t0, t1 = {"whole": (0, 1), "wide": (a, b), "narrow": (a, a + (1 - a) / 64), "at 0": (0, b / 16),
                  "at 1": (1 - b / 16, 1)}[box]
        t0, t1, s = np.float32(t0), np.float32(t1), np.float32(rng.random())
        x = float(s) * cdf(float(t1)) + (1 - float(s)) * cdf(float(t0))
        lo, hi = float(t0), float(t1)
        for _ in range(60):
            m = 0.5 * (lo + hi)
            lo, hi = (m, hi) if cdf(m) < x else (lo, m)
        tol = 16 * 2.0 ** -24 * cdf(1.0) / low + 2.0 ** -23
        assert abs(_draw(s, t0, t1, q) - lo) <= tol, (q, t0, t1, s)
        checked += 1


@pytest.mark.parametrize("p", [(0, 0, 0), (0, 1, 0), (1, 0, 1), (0, 0, 1), (1, 0, 0), (1e-38, 2e-38, 1e-38),
                               (3e37, 1e37, 3e37), (np.inf, 1, 1), (np.nan, 1, 1), (-1, -1, -1)], ids=str)
def test_draw_stays_in_the_box(p):
    for t0, t1 in [(0.0, 1.0), (0.0, 0.0), (1.0, 1.0), (0.25, 0.25), (0.25, 0.5), (0.0, 1e-6), (0.999999, 1.0)]:
        for s in (0.0, 1e-7, 0.3, 0.5, 0.9999999):
            t0f, t1f = float(np.float32(t0)), float(np.float32(t1))
            r = _draw(s, t0f, t1f, p)
            assert t0f <= r <= np.nextafter(np.float32(t1f), np.float32(2)), (t0, t1, s, r)
