"""GPU: FP64 matmul of the scalar kernels where points of one leaf lie far
apart, against the oracle to 1e-12.  Two groups of 110 points share a leaf of
up to 300 although they are 8e4 (8e6) lengthscales apart: distances that are
right within a group need coordinate differences, since a distance expanded
into squares and a product loses the square of the leaf's extent."""
import numpy as np
import pytest

import oracle as O
from h2pack_amd import construct as C
from h2pack_amd.h2mat import H2MatHIP
from tests.problems import rel

pytestmark = pytest.mark.gpu


# (Matern at 1e7: the construction's interpolation overflows, its bases hold
# infinities and the oracle's product is NaN)
@pytest.mark.parametrize("kid,par,gap", [(C.KRNL_GAUSSIAN, [1.0], 1e5), (C.KRNL_MATERN32, [1.0], 1e5),
                                         (C.KRNL_COULOMB, [], 1e5), (C.KRNL_GAUSSIAN, [1.0], 1e7),
                                         (C.KRNL_COULOMB, [], 1e7)])
def test_leaf_of_distant_groups_matches_oracle(kid, par, gap):
    rng = np.random.default_rng(41)
    a, b = rng.random((3, 110)) * 2.0, rng.random((3, 110)) * 2.0
    a[:2] += [[3 * gap], [2.2 * gap]]
    b[:2] += [[3 * gap], [3 * gap]]
    coord = np.concatenate([rng.random((3, 1500)) * 6.0, a, b], axis=1)
    h2 = C.build_h2(coord, kid, par, 1e-8, 300, BD_JIT=1, pp_kind="surface", host_blocks=False)
    pts = np.asarray(h2.coord).reshape(3, -1)
    wide = max(np.ptp(pts[:, h2.pt_cluster[2 * k]:h2.pt_cluster[2 * k + 1] + 1], axis=1).max() for k in h2.leaf_nodes)
    assert wide > 0.7 * gap                  # the groups share a leaf
    X = rng.standard_normal((h2.krnl_mat_size, 20))
    ref = O.OracleH2(h2, BD_JIT=1).matmul(X, "col", n_thread=8)
    m = H2MatHIP(h2, mode="jit")
    for n_vec in (3, 20):
        err = rel(m.matmul(X[:, :n_vec], "col"), ref[:, :n_vec])
        print(f"[leaf extent {wide:.0f}, kernel {kid}, {n_vec} columns] {err:.2e}", flush=True)
        assert err < 1e-12
    m.close()
