"""The FP32 square root of the FP32-mixed matmul (sqrt_from_rsq), compiled for
the host from the device header and given emulated estimates of 1/sqrt(q).

With an estimate off by a relative d, the correction leaves d^2 terms (below
2^-40 for one unit in the last place) beside the final rounding: 1/2 + 2^-18
units.  From q = 2^-102 down the residual q - s^2 is rounded to a multiple of
2^-149 (half of one, times y/2 <= 2^62: a quarter unit of s more)."""
import ctypes as ct
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HDR = os.path.join(ROOT, "h2pack_amd", "csrc", "h2p_exp2.h")

SRC = r"""
#include "h2p_exp2.h"
extern "C" void roots(const float *q, const float *y, float *s, long n) {
    for (long i = 0; i < n; i++) s[i] = h2p::sqrt_from_rsq(q[i], y[i]);
}
"""


@pytest.fixture(scope="module")
def roots(tmp_path_factory):
    d = tmp_path_factory.mktemp("sqrtq")
    (d / "s.cpp").write_text(SRC)
    so = d / "libs.so"
    subprocess.run(["g++", "-O2", "-mfma", "-ffp-contract=off", "-fPIC", "-shared", "-I", os.path.dirname(HDR),
                    "-o", str(so), str(d / "s.cpp")], check=True)
    L = ct.CDLL(str(so))
    L.roots.argtypes = [ct.c_void_p, ct.c_void_p, ct.c_void_p, ct.c_long]
    L.roots.restype = None

    def f(q, y):
        s = np.empty_like(q)
        L.roots(q.ctypes.data, y.ctypes.data, s.ctypes.data, q.size)
        return s
    return f


def estimate(q, ulps):
    """1/sqrt(q) rounded to FP32, then moved by whole units in the last place."""
    y = (1.0 / np.sqrt(q.astype(np.float64))).astype(np.float32)
    return (y.view(np.int32) + np.int32(ulps)).view(np.float32)


@pytest.mark.parametrize("ulps", [0, 1, -1])
def test_every_mantissa(roots, ulps):
    q = np.arange(0x3f800000, 0x40800000, dtype=np.int32).view(np.float32)   # [1, 4)
    s = roots(q, estimate(q, ulps))
    r = np.sqrt(q.astype(np.float64))
    ulp = np.where(r < 2.0, 2.0 ** -23, 2.0 ** -22)
    assert np.max(np.abs(s - r) / ulp) <= 0.5 + 2.0 ** -18
    if ulps == 0:
        assert np.array_equal(s, r.astype(np.float32))


@pytest.mark.parametrize("ulps", [0, 1, -1])
def test_small_and_zero(roots, ulps):
    rng = np.random.default_rng(2)
    q = rng.integers(0x00800000, 0x0c800000, 2_000_000, dtype=np.int32).view(np.float32)   # 2^-126 .. 2^-102
    s = roots(q, estimate(q, ulps))
    r = np.sqrt(q.astype(np.float64))
    ulp = np.exp2(np.floor(np.log2(r)) - 23)
    assert np.max(np.abs(s - r) / ulp) <= 0.75 + 2.0 ** -18
    # zero and subnormals, whose estimate the hardware gives as infinity
    q = np.concatenate([[0], rng.integers(1, 0x00800000, 1000, dtype=np.int32)]).astype(np.int32).view(np.float32)
    s = roots(q, np.full(q.size, np.inf, np.float32))
    assert s[0] == 0.0 and np.all((s >= 0.0) & (s <= 2.0 ** -63))
