"""The matvec kernels' exponential (exp2_neg128x, both halves), compiled for the
host from the device header.

It is exp2_neg128 (whose accuracy test_exp2.py pins) with the exponent added
by an integer instead of ldexp: where the result is a normal number the two
are the same bits.  Subnormal results of the clamped form are rounded once more
(half a subnormal unit), and it is 0 from 2^-1075 on, for +inf too."""
import ctypes as ct
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HDR = os.path.join(ROOT, "h2pack_amd", "csrc", "h2p_exp2.h")

SRC = r"""
#include "h2p_exp2.h"
static const double tab[H2P_E2_N] = {H2P_E2_TABLE};
template <bool F> static double one(double x, const double *t) {
    return h2p::exp2_neg128x_end<F>(h2p::exp2_neg128x_begin<F>(x, t), H2P_E2X_C2);
}
extern "C" void base(const double *x, double *y, long n) {
    for (long i = 0; i < n; i++) y[i] = h2p::exp2_neg128(x[i], tab);
}
extern "C" void ex(const double *x, double *y, long n, int fast) {
    double t[H2P_E2_N];
    for (int j = 0; j < H2P_E2_N; j++) t[j] = h2p::e2x_entry(tab[j], j);
    for (long i = 0; i < n; i++) y[i] = fast ? one<true>(x[i], t) : one<false>(x[i], t);
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("exp2x")
    (d / "e.cpp").write_text(SRC)
    so = d / "libe.so"
    subprocess.run(["g++", "-O2", "-mfma", "-ffp-contract=off", "-fPIC", "-shared", "-I", os.path.dirname(HDR),
                    "-o", str(so), str(d / "e.cpp")], check=True)
    L = ct.CDLL(str(so))
    L.ex.argtypes = [ct.c_void_p, ct.c_void_p, ct.c_long, ct.c_int]
    L.ex.restype = None
    L.base.argtypes = [ct.c_void_p, ct.c_void_p, ct.c_long]
    L.base.restype = None
    return L


def run(lib, x, fast):
    x = np.ascontiguousarray(x, dtype=np.float64)
    y = np.empty_like(x)
    lib.ex(x.ctypes.data, y.ctypes.data, x.size, int(fast))
    return y


@pytest.mark.parametrize("fast", [True, False])
@pytest.mark.parametrize("top", [1.0, 64.0, 1000.0])
def test_same_bits_as_the_plain_form(lib, fast, top):
    rng = np.random.default_rng(3)
    x = np.concatenate([rng.random(400_000) * top * 128, np.arange(0, 512) / 4.0, [-1e-11, 0.0, top * 128]])
    y = np.empty_like(x)
    lib.base(x.ctypes.data, y.ctypes.data, x.size)
    assert np.array_equal(run(lib, x, fast), y)


def test_underflow_and_beyond(lib):
    x = np.concatenate([np.linspace(1000, 1074.9, 20001), [1075.5, 1099.0, 1200.0, 1e30, np.inf]]) * 128
    y = run(lib, x, False)
    ref = np.exp2(-x[:-5].astype(np.longdouble) / 128)
    assert np.all(np.abs(y[:-5] - ref) <= ref * 3.5e-16 + np.longdouble(2) ** -1075)
    assert np.all(y[-5:] == 0.0)
