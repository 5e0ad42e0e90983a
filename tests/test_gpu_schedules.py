"""GPU: the matvec schedules of JIT handles pinned one by one.  Small handles
(fewer than 2.5e8 kernel pairs) run in order with all blocks in one launch by
default; larger ones run their D blocks on a second stream beside the sweeps
and their leaf outputs in two launches.  Both kinds on small matrices: every
one gives bitwise the y of the profiled path, which runs each launch in order
on one stream."""
import numpy as np
import pytest

from h2pack_amd.h2mat import H2MatHIP
from tests.problems import problem

pytestmark = pytest.mark.gpu

SCALAR = [("gaussian", "fp64"), ("coulomb", "fp64"), ("matern32", "fp64"), ("gaussian", "fp32mix"),
          ("matern32", "fp32mix")]


def handle(name, prec, monkeypatch, graph=True):
    if not graph:
        monkeypatch.setenv("H2P_HIP_NO_GRAPH", "1")
    m = H2MatHIP(problem(name)[0], mode="jit", prec=prec)
    if not graph:
        monkeypatch.delenv("H2P_HIP_NO_GRAPH")
    return m


def in_order(m, x):
    m.set_profiling(True)
    y = m.matvec(x)
    info = m.info()
    m.set_profiling(False)
    return y, info


@pytest.mark.parametrize("d_late", [None, "0", "1"])
@pytest.mark.parametrize("name,prec", SCALAR)
def test_concurrent_d_blocks_agree(name, prec, d_late, monkeypatch):
    """D blocks on the second stream, part of them after the B blocks
    (H2P_HIP_D_LATE: the default, none, all), eagerly and at the default share
    as a graph."""
    import torch
    if d_late is not None:
        monkeypatch.setenv("H2P_HIP_D_LATE", d_late)
    ms = [handle(name, prec, monkeypatch, graph=False)]
    if d_late is None:
        ms.append(handle(name, prec, monkeypatch))
    rng = np.random.default_rng(23)
    junk = torch.randn(1 << 20, device="cuda:0", dtype=torch.float64)
    for k in (0, 2):
        for m in ms:
            m.mm_variant(5, 0, k)
            assert m.info()["mv_d_concurrent"] == 1
        for it in range(2):
            x = rng.random(ms[0].N) - 0.5
            y_serial, info = in_order(ms[0], x)
            assert info["t_blocks_d"] > 0.0 and info["t_blocks_b"] > 0.0
            for m in ms:
                y = m.matvec(x)
                junk.mul_(1.0001).add_(0.5)
                torch.cuda.synchronize()
                assert np.array_equal(y, y_serial), (k, it)
    for m in ms:
        m.close()


@pytest.mark.parametrize("name,prec", SCALAR)
def test_default_of_small_handles_agrees(name, prec, monkeypatch):
    """All blocks in one launch, in order, as a graph and eagerly."""
    for graph in (True, False):
        m = handle(name, prec, monkeypatch, graph)
        info = m.info()
        assert info["mv_d_concurrent"] == 0 and info["mv_level_split"] == 0
        x = np.random.default_rng(24).random(m.N) - 0.5
        for it in range(2):
            assert np.array_equal(m.matvec(x), in_order(m, x)[0]), (graph, it)
        m.close()


@pytest.mark.parametrize("schedule", [0, 2, 3])
def test_graph_follows_caller_pointers_in_every_schedule(schedule, monkeypatch):
    """Replays of the captured matvec alternating between x and y buffers:
    its gather and its last launch (the leaf outputs' second one where D
    blocks run beside the sweeps) are pointed at them."""
    import torch
    m = handle("gaussian", "fp64", monkeypatch)
    m.mm_variant(5, 0, schedule)
    rng = np.random.default_rng(31)
    xs = [torch.from_numpy(rng.random(m.N) - 0.5).to("cuda:0") for _ in range(3)]
    ys = [torch.full((m.N,), np.nan, dtype=torch.float64, device="cuda:0") for _ in range(3)]
    ref = [in_order(m, x.cpu().numpy())[0] for x in xs]
    for i, j in [(0, 0), (1, 1), (2, 2), (0, 1), (2, 0), (1, 2), (0, 0)]:
        before = [y.cpu().numpy() for y in ys]
        m.matvec_dev(xs[i].data_ptr(), ys[j].data_ptr())
        torch.cuda.synchronize()
        for k in range(3):
            assert np.array_equal(ys[k].cpu().numpy(), ref[i] if k == j else before[k], equal_nan=True), (i, j, k)
    m.close()


@pytest.mark.parametrize("name", ["gaussian", "coulomb", "matern32"])
def test_fp64_occupancy_build_agrees(name, monkeypatch):
    """The FP64 block launch compiled without an occupancy target (variant 1,
    which the tuner may choose), launched eagerly in order: same bits as the
    default build, in one launch and in parts."""
    m = handle(name, "fp64", monkeypatch, graph=False)
    x = np.random.default_rng(5).random(m.N) - 0.5
    y = m.matvec(x)
    m.mm_variant(4, 1, 1)
    assert m.mm_variant(4, 1) == 1
    assert np.array_equal(m.matvec(x), y)
    assert np.array_equal(in_order(m, x)[0], y)
    m.close()


@pytest.mark.parametrize("name", ["gaussian", "rpy"])
def test_matmul_graph_is_recaptured_for_the_other_task_order(name, monkeypatch):
    """Changing a phase's task order drops the captured product phases; the
    replays before and after equal an eager handle's bit for bit."""
    import torch
    g, e = handle(name, "fp64", monkeypatch), handle(name, "fp64", monkeypatch, graph=False)
    rng = np.random.default_rng(22)
    junk = torch.randn(1 << 20, device="cuda:0", dtype=torch.float64)
    for it in range(6):
        if it % 2 == 0:
            g.mm_variant(-1, 8, 1 - g.mm_variant(-1, 8))
        X = rng.standard_normal((g.N, 8))
        Y = g.matmul(X, "col")
        junk.mul_(1.0001).add_(0.5)
        torch.cuda.synchronize()
        assert np.array_equal(Y, e.matmul(X, "col")), it
    g.close()
    e.close()
