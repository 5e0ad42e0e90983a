"""GPU: the matvec tuner's shared choices keep apart handles that have the list
of all blocks in one launch and handles that do not: "in order" is another
schedule on each.  Two trees of one point sequence, whose block histograms are
the same, on either side of the limit of 2.5e8 kernel pairs."""
import numpy as np
import pytest

from h2pack_amd import construct as C
from h2pack_amd.h2mat import H2MatHIP

pytestmark = pytest.mark.gpu


def build(n):
    coord = np.random.default_rng(77).random((3, 90_000))[:, :n] * 20.0
    return C.build_h2(coord, C.KRNL_MATERN32, [1.0], 1e-4, 300, BD_JIT=1, pp_kind="surface", host_blocks=False)


def histogram(h2):
    h = {}
    for nr, nc in list(zip(h2.B_nrow, h2.B_ncol)) + list(zip(h2.D_nrow, h2.D_ncol)):
        if nr * nc:
            k = (int(np.log2(nr)), int(np.log2(nc)))
            h[k] = h.get(k, 0) + 1
    return {k: int(np.log2(v)) for k, v in h.items()}


def test_choices_are_not_shared_across_the_limit():
    small, large = build(59_100), build(59_500)
    assert histogram(small) == histogram(large)
    a, a2, b = (H2MatHIP(h, mode="jit", prec="fp32mix") for h in (small, small, large))
    assert a.info()["mv_d_concurrent"] == 0 and b.info()["mv_d_concurrent"] == 1   # the defaults on either side
    ta, ta2, tb = a.autotune(0), a2.autotune(0), b.autotune(0)
    print(f"small {ta} large {tb}", flush=True)
    assert ta["default_ms"] > 0.0
    assert ta2["default_ms"] == 0.0 and ta2["d_concurrent"] == ta["d_concurrent"]   # taken from the cache
    assert tb["default_ms"] > 0.0                                                   # timed on its own blocks
    for m, h2 in ((a, small), (b, large)):
        x = np.random.default_rng(3).random(h2.krnl_mat_size) - 0.5
        y = m.matvec(x)
        m.set_profiling(True)
        assert np.array_equal(y, m.matvec(x))
        m.set_profiling(False)
        m.close()
    a2.close()
