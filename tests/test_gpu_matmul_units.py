"""GPU: FP32-mixed Matern matmul in small units of length (l grows as the
coordinates shrink, the kernel values stay the same): squared distances far
below 1e-30 and the zero ones of the diagonal, against the oracle to the
FP32-mixed bar of 1e-6, and the matvec of the same handle with it."""
import numpy as np
import pytest

import oracle as O
from h2pack_amd import construct as C
from h2pack_amd.h2mat import H2MatHIP
from tests.problems import rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("unit", [1.0, 1e-12, 1e-16])
def test_small_units_match_oracle(unit):
    rng = np.random.default_rng(6)
    coord = rng.random((3, 1200)) * (4.0 * unit)
    h2 = C.build_h2(coord, C.KRNL_MATERN32, [1.0 / unit], 1e-8, 60, BD_JIT=1, pp_kind="surface", host_blocks=False)
    X = rng.standard_normal((h2.krnl_mat_size, 8))
    ref = O.OracleH2(h2, BD_JIT=1).matmul(X, "col", n_thread=8)
    m = H2MatHIP(h2, mode="jit", prec="fp32mix")
    err, err_mv = rel(m.matmul(X, "col"), ref), rel(m.matvec(X[:, 0].copy()), ref[:, 0])
    print(f"[unit {unit:g}] matmul {err:.2e} matvec {err_mv:.2e}", flush=True)
    assert err < 1e-6 and err_mv < 1e-6
    m.close()
