"""The Simpson rule's division by 6 as a product corrected by its exact remainder
(csrc/region_math.h): the quotient bit for bit, compiled for the host as the kernels'
arithmetic is."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = """
#include "viltrum_amd/csrc/region_math.h"
extern "C" void simpson_d(long n, const double* p, double* o) { for (long i = 0; i < n; ++i) o[i] = vmx::simpson(p[3 * i], p[3 * i + 1], p[3 * i + 2]); }
extern "C" void simpson_f(long n, const float* p, float* o) { for (long i = 0; i < n; ++i) o[i] = vmx::simpson(p[3 * i], p[3 * i + 1], p[3 * i + 2]); }
extern "C" void metric_f(long n, const float* p, float* o) { for (long i = 0; i < n; ++i) o[i] = vmx::metric_relative(p[3 * i], p[3 * i + 1]); }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("division")
    src, out = str(d / "s.cpp"), str(d / "s.so")
    with open(src, "w") as f:
        f.write(SRC)
    subprocess.run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-ffp-contract=off", "-I", ROOT, "-o", out, src],
                   check=True)
    return C.CDLL(out)


def _call(fn, p, dt):
    o = np.zeros(len(p), dtype=dt)
    fn(C.c_long(len(p)), p.ctypes.data_as(C.c_void_p), o.ctypes.data_as(C.c_void_p))
    return o


def _triples(dt, bits, seed):
    """Random bit patterns (every exponent, infinities, NaN, zeros of both signs)."""
    rng = np.random.default_rng(seed)
    p = rng.integers(0, 1 << bits, 600000, dtype=np.uint64 if bits == 64 else np.uint32).view(dt).reshape(-1, 3).copy()
    special = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1.0, -1.0, 6.0, np.finfo(dt).max, np.finfo(dt).tiny,
                        np.nextafter(dt(0), dt(1))], dtype=dt)
    p[:30000] = special[rng.integers(0, len(special), (30000, 3))]
    p[30000:60000] = rng.standard_normal((30000, 3)).astype(dt)
    return np.ascontiguousarray(p)


def _same(a, b):
    return np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~np.isnan(a)].view(np.uint8),
                                                                       b[~np.isnan(b)].view(np.uint8))


@pytest.mark.parametrize("dt,bits,fn", [(np.float32, 32, "simpson_f"), (np.float64, 64, "simpson_d")])
def test_simpson_is_the_quotient(lib, dt, bits, fn):
    p = _triples(dt, bits, 1)
    with np.errstate(all="ignore"):
        q = p.astype(np.float64)
        want = ((q[:, 0] + 4.0 * q[:, 1] + q[:, 2]) / 6.0).astype(dt)
    assert _same(_call(getattr(lib, fn), p, dt), want)


def test_relative_metric_threshold(lib):
    """The FP32 threshold 1e-37 is compared in FP32: the neighbours of it, and random bits."""
    p = _triples(np.float32, 32, 2)
    t = np.float32(1e-37)
    near = np.array([np.nextafter(t, np.float32(0)), t, np.nextafter(t, np.float32(1))], dtype=np.float32)
    p[60000:60009, 0] = np.repeat(near, 3)
    p[60000:60009, 1] = np.tile(near, 3)
    with np.errstate(all="ignore"):
        a, b = p[:, 0], p[:, 1]
        ma = np.where(np.abs(a) < np.abs(b), np.abs(b), np.abs(a))
        want = np.where(ma.astype(np.float64) < 1e-37, np.abs(b - a), np.abs(b - a) / ma)
    assert _same(_call(lib.metric_f, p, np.float32), want.astype(np.float32))
