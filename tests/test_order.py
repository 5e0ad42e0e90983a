"""The one-launch list of a handle's block tasks (merge_parts), compiled for the
host: the list that a stable sort of the parts by work and a stable partition
into workgroup and wave tasks give, in a number of comparisons linear in the
tasks."""
import ctypes as ct
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HDR = os.path.join(ROOT, "h2pack_amd", "csrc", "h2p_order.h")

SRC = r"""
#include "h2p_order.h"
struct T { long work, wave, id; };
// parts end at end[0 .. np); tasks are ordered within their part first.
// Returns the comparisons of merge_parts, or -1 if the two lists differ.
extern "C" long check(const long *work, const long *wave, const int *end, int np, long *nbig) {
    std::vector<T> t;
    std::vector<h2p::PartRange> parts;
    long cmp = 0;
    auto more = [&](const T &x, const T &y) { cmp++; return x.work > y.work; };
    for (int p = 0, b = 0; p < np; b = end[p++]) {
        for (int i = b; i < end[p]; i++) t.push_back({work[i], wave[i], i});
        std::stable_sort(t.begin() + b, t.end(), more);
        auto m = std::stable_partition(t.begin() + b, t.end(), [](const T &x) { return !x.wave; });
        parts.push_back({b, (int)(m - (t.begin() + b)), end[p] - b});
    }
    std::vector<T> ref = t;
    std::stable_sort(ref.begin(), ref.end(), more);
    const long rbig =
        std::stable_partition(ref.begin(), ref.end(), [](const T &x) { return !x.wave; }) - ref.begin();
    cmp = 0;
    int big = -1;
    const std::vector<T> out = h2p::merge_parts(t, parts, more, &big);
    *nbig = big;
    if (big != rbig || out.size() != ref.size()) return -1;
    for (size_t i = 0; i < out.size(); i++)
        if (out[i].id != ref[i].id) return -1;
    return cmp;
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("order")
    (d / "o.cpp").write_text(SRC)
    so = d / "libo.so"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-I", os.path.dirname(HDR), "-o", str(so),
                    str(d / "o.cpp")], check=True)
    L = ct.CDLL(str(so))
    L.check.argtypes = [ct.c_void_p, ct.c_void_p, ct.c_void_p, ct.c_int, ct.c_void_p]
    L.check.restype = ct.c_long
    return L


@pytest.mark.parametrize("sizes", [(0, 0, 0), (1, 0, 0), (0, 3, 1), (7, 7, 7), (5000, 40, 9000), (0, 0, 20_000)])
@pytest.mark.parametrize("distinct", [3, 1000])      # many and few equal works
@pytest.mark.parametrize("limit", [-1, 400, 2000])   # no wave tasks, some, all
def test_merged_list_is_the_sorted_one(lib, sizes, distinct, limit):
    rng = np.random.default_rng(sum(sizes) + distinct)
    n = sum(sizes)
    work = rng.integers(1, distinct + 1, n).astype(np.int64)
    wave = (rng.integers(0, 1001, n) < limit).astype(np.int64)
    end = np.cumsum(sizes).astype(np.int32)
    nbig = np.zeros(1, np.int64)
    cmp = lib.check(work.ctypes.data, wave.ctypes.data, end.ctypes.data, len(sizes), nbig.ctypes.data)
    assert 0 <= cmp <= 2 * n
    assert nbig[0] == n - wave.sum()
