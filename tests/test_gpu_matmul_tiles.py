"""GPU: the matmul kernels at the edges of their tiles, against the oracle.

Tasks hold up to 32 rows (16 points for the evaluated 3x3 kernel), their
inner entries go in chunks of 16 dealt to four waves, columns in tiles of 16
(one to four per chunk of 64): column counts around every tile width, trees
whose ranks and leaves leave ragged pieces, fewer chunks than waves, and a
point set so wide that the exponential's argument is clamped.  Bars as in
the other parity tests: FP64 1e-12, FP32-mixed 1e-6.
"""
import numpy as np
import pytest

import oracle as O
from h2pack_amd import construct as C
from h2pack_amd.h2mat import H2MatHIP
from tests.problems import problem, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["tiny_coulomb", "tiny_gaussian", "matern32", "tiny_rpy", "hss_gaussian"])
@pytest.mark.parametrize("mode", ["jit", "aot"])
def test_column_tiles_match_oracle(name, mode):
    h2, _ = problem(name)
    rng = np.random.default_rng(31)
    X = rng.standard_normal((h2.krnl_mat_size, 66))
    ref = O.OracleH2(h2, BD_JIT=1).matmul(X, "col", n_thread=8)
    handles = [(H2MatHIP(h2, mode=mode, host_blocks=False), 1e-12)]
    if h2.krnl_dim == 1:
        handles.append((H2MatHIP(h2, mode=mode, prec="fp32mix", host_blocks=False), 1e-6))
    for m, bar in handles:
        for n_vec in (1, 15, 16, 17, 33, 48, 49, 64, 66):
            for layout in ("col", "row"):
                err = rel(m.matmul(X[:, :n_vec], layout), ref[:, :n_vec])
                assert err < bar, (n_vec, layout, err)
        m.close()


@pytest.mark.parametrize("kid", [C.KRNL_GAUSSIAN, C.KRNL_MATERN32])
def test_wide_point_set_matches_oracle(kid):
    """Two clusters 1e6 lengthscales apart: the distances between them take
    the exponential far past its range, inside the clusters it is ordinary."""
    rng = np.random.default_rng(7)
    coord = rng.random((3, 700)) * 4.0
    coord[0, 350:] += 1e6
    h2 = C.build_h2(coord, kid, [1.0], 1e-8, 60, BD_JIT=1, pp_kind="surface", host_blocks=False)
    X = rng.standard_normal((h2.krnl_mat_size, 20))
    ref = O.OracleH2(h2, BD_JIT=1).matmul(X, "col", n_thread=8)
    Y = H2MatHIP(h2, mode="jit").matmul(X, "col")
    # coordinates of 1e6 leave differences 1e-10 absolute: the bar is theirs
    assert np.isfinite(Y).all() and rel(Y, ref) < 1e-9


@pytest.mark.parametrize("kid", [C.KRNL_GAUSSIAN, C.KRNL_MATERN32])
@pytest.mark.parametrize("scale", [1.0, 12.0, 60.0])
def test_matvec_underflowing_blocks_match_oracle(kid, scale):
    """Blocks whose kernel values stay normal take the short exponential, those
    that can underflow the other: trees with none, some and many of the latter."""
    rng = np.random.default_rng(8)
    coord = rng.random((3, 3000)) * 6.0 * scale
    h2 = C.build_h2(coord, kid, [1.0], 1e-8, 90, BD_JIT=1, pp_kind="surface", host_blocks=False)
    x = rng.random(h2.krnl_mat_size) - 0.5
    ref = O.OracleH2(h2, BD_JIT=1).matvec(x, n_thread=8)
    m = H2MatHIP(h2, mode="jit")
    assert rel(m.matvec(x), ref) < 1e-12
    m.close()
