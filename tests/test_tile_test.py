"""The tile test's division by a known divisor against IEEE division, bit for
bit, on the host: ordinary operands, quotients near rounding midpoints, and
operands outside the range of the shortcut (zero, subnormal, huge, infinite,
NaN)."""
import ctypes as C
import os

import numpy as np

from tinygs_amd import _lib

import pytest


def _quotients(a, c):
    if not os.path.exists(_lib.LIB_PATH):
        pytest.skip("library not built")
    f = getattr(_lib.load(), "_ZN3tgs19tile_test_quotientsEPKfS1_Pfl")
    p = C.POINTER(C.c_float)
    f.argtypes, f.restype = [p, p, p, C.c_int64], None
    a, c = np.ascontiguousarray(a, np.float32), np.ascontiguousarray(c, np.float32)
    out = np.empty_like(a)
    f(a.ctypes.data_as(p), c.ctypes.data_as(p), out.ctypes.data_as(p), a.size)
    return out


def _check(a, c):
    a, c = np.asarray(a, np.float32), np.asarray(c, np.float32)
    with np.errstate(all="ignore"):
        ref = a / ((np.float32(15.0) * c) * np.float32(15.0))
    got = _quotients(a, c)
    same = (got.view(np.uint32) == ref.view(np.uint32)) | (np.isnan(got) & np.isnan(ref))
    assert same.all(), (a[~same][:4], c[~same][:4], got[~same][:4], ref[~same][:4])


def test_random_operands():
    rng = np.random.default_rng(0)
    n = 1 << 20
    for lo, hi in ((-3, 3), (-60, 60), (-149, 127)):
        sign = np.where(rng.random(n) < 0.5, -1.0, 1.0)
        a = sign * np.ldexp(1.0 + rng.random(n), rng.integers(lo, hi, n))
        c = np.ldexp(1.0 + rng.random(n), rng.integers(max(lo, -40), min(hi, 40), n))
        _check(a.astype(np.float32), c.astype(np.float32))


def test_quotients_near_midpoints():
    rng = np.random.default_rng(1)
    n = 1 << 20
    c = np.ldexp(1.0 + rng.random(n), rng.integers(-12, 3, n)).astype(np.float32)
    b = (np.float32(15.0) * c) * np.float32(15.0)
    q = (1.0 + rng.random(n)).astype(np.float32)
    mid = q.astype(np.float64) + np.ldexp(1.0, -24)   # halfway to the next float in [1, 2)
    a = (mid * b).astype(np.float32)
    for step in (-1, 0, 1):
        _check((a.view(np.int32) + step).view(np.float32), c)


def test_special_operands():
    v = np.array([0.0, -0.0, 1.0, -1.0, 1e-45, 1e-38, 1.2e-38, 1e-30, 1e30, 3.4e38, np.inf, -np.inf, np.nan,
                  2.0**-60, 2.0**60, 2.0**-48, 2.0**33], np.float32)
    a, c = np.meshgrid(v, v)
    _check(a.reshape(-1), c.reshape(-1))
