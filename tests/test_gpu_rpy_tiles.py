"""GPU: the tiled RPY launch at its edges, against the oracle to 1e-12:
blocks narrower and wider than the limit of a wave unit (96 points), targets
in one and several staged chunks (64 points), sources in one and several
passes, and unequal radii with overlapping, touching and separated spheres
in the same tree (the blocks known to be far take the tensor's far form)."""
import numpy as np
import pytest

import oracle as O
from h2pack_amd import construct as C
from h2pack_amd.h2mat import H2MatHIP
from tests.problems import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("leaf", [24, 70, 110, 260])
@pytest.mark.parametrize("radii", ["equal", "unequal"])
def test_rpy_tiles_match_oracle(leaf, radii):
    n = 2000
    rng = np.random.default_rng(17)
    side = (n * (4.0 / 3.0) * np.pi / 0.15) ** (1.0 / 3.0)
    a = np.ones((1, n)) if radii == "equal" else rng.uniform(0.3, 1.5, (1, n))
    coord = np.concatenate([rng.random((3, n)) * side, a], axis=0)
    coord[:3, 1] = coord[:3, 0] + np.array([a[0, 0] + a[0, 1], 0.0, 0.0])   # touching
    h2 = C.build_h2(coord, C.KRNL_RPY, [1.0], 1e-7, leaf, BD_JIT=1, pp_kind="surface", host_blocks=False)
    x = rng.random(h2.krnl_mat_size) - 0.5
    X = rng.standard_normal((h2.krnl_mat_size, 5))
    orc = O.OracleH2(h2, BD_JIT=1)
    m = H2MatHIP(h2, mode="jit")
    err, err_mm = rel(m.matvec(x), orc.matvec(x, n_thread=8)), rel(m.matmul(X, "col"), orc.matmul(X, "col", n_thread=8))
    print(f"[rpy leaf={leaf} {radii}] matvec {err:.2e} matmul {err_mm:.2e}, largest leaf "
          f"{max(h2.pt_cluster[2 * k + 1] - h2.pt_cluster[2 * k] + 1 for k in h2.leaf_nodes)}, "
          f"ranks to {max(h2.U_ncol) // 3}", flush=True)
    assert err < 1e-12 and err_mm < 1e-12
    m.close()
