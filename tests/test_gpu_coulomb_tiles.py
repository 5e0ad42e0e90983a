"""GPU: the tiled FP64 Coulomb launch at its edges, against the oracle to
1e-12: leaves from a fraction of a 16-point tile to more than a wave unit's
80 targets and a pass's 128 sources, and coincident points, inside a leaf and
in neighbouring leaves, whose entries are the kernel's diagonal value."""
import numpy as np
import pytest

import oracle as O
from h2pack_amd import construct as C
from h2pack_amd.h2mat import H2MatHIP
from tests.problems import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("leaf", [9, 33, 85, 135, 300])
@pytest.mark.parametrize("diag", [[], [2.5]])
def test_coulomb_tiles_match_oracle(leaf, diag):
    n = 2500
    rng = np.random.default_rng(23)
    coord = rng.random((3, n)) * 13.0
    coord[:, 0] = coord[:, 1]          # coincident pairs
    coord[:, 2:40] = coord[:, 40:78]
    h2 = C.build_h2(coord, C.KRNL_COULOMB, diag, 1e-6, leaf, BD_JIT=1, pp_kind="surface", host_blocks=False)
    x = rng.random(n) - 0.5
    m = H2MatHIP(h2, mode="jit")
    err = rel(m.matvec(x), O.OracleH2(h2, BD_JIT=1).matvec(x, n_thread=8))
    print(f"[coulomb leaf={leaf} diag={diag}] {err:.2e}", flush=True)
    assert err < 1e-12
    m.close()
