"""GPU: the sweeps, skeleton sums and leaf outputs at every chunk width they
choose (256, 64 and 16 outputs a workgroup, by the number of nodes and rows of
a launch), leaves that sum their own partials and leaves that do not, ranks
and rows that are no multiple of a chunk; against the oracle to 1e-12."""
import numpy as np
import pytest

import oracle as O
from h2pack_amd import construct as C
from h2pack_amd.h2mat import H2MatHIP
from tests.problems import rel

pytestmark = pytest.mark.gpu


# few nodes (16 wide), one level (leaves sum their own), hundreds of nodes
# (64 wide), thousands of leaves of a few points (256 wide)
@pytest.mark.parametrize("kernel,n,leaf,mode", [
    ("gaussian", 1501, 60, "aot"), ("gaussian", 4003, 150, "jit"), ("gaussian", 9001, 5, "aot"),
    ("coulomb", 9001, 40, "jit"), ("coulomb", 12_007, 60, "aot"),
    ("rpy", 700, 40, "jit"), ("rpy", 3001, 12, "jit"), ("rpy", 5003, 3, "aot"),
])
def test_sweep_widths_match_oracle(kernel, n, leaf, mode):
    rng = np.random.default_rng(31)
    if kernel == "rpy":
        side = (n * (4.0 / 3.0) * np.pi / 0.1) ** (1.0 / 3.0)
        coord = np.concatenate([rng.random((3, n)) * side, np.ones((1, n))])
        h2 = C.build_h2(coord, C.KRNL_RPY, [1.0], 1e-6, leaf, BD_JIT=1, pp_kind="surface", host_blocks=False)
    else:
        coord = C.uniform_cube_points(n, 10.0, 31)
        kid, par = (C.KRNL_GAUSSIAN, [1.0]) if kernel == "gaussian" else (C.KRNL_COULOMB, [])
        h2 = C.build_h2(coord, kid, par, 1e-6, leaf, BD_JIT=1, pp_kind="surface", host_blocks=False)
    x = rng.random(h2.krnl_mat_size) - 0.5
    m = H2MatHIP(h2, mode=mode, host_blocks=False)
    err = rel(m.matvec(x), O.OracleH2(h2, BD_JIT=1).matvec(x, n_thread=8))
    print(f"[{kernel} n={n} leaf={leaf} {mode}] {err:.2e}", flush=True)
    assert err < 1e-12
    m.close()
