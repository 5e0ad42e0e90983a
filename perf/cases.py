"""Performance cases: the applies that a user of this framework runs, through
its public entry points (``H2MatHIP`` and ``H2Batch``), on one GPU.

A case is a dict of plain values:

  op       "matvec", "matmul", "cg" (a co-scheduled batch of CG solves)
  kernel   "coulomb", "gaussian", "matern32", "rpy", "rpy_periodic"
  n        points; density (points per unit volume, or the particles' volume
           fraction for RPY), l (the kernel parameter), leaf, reltol
  mode     "jit" or "aot" (blocks evaluated on the device at upload)
  prec     "fp64" or "fp32mix"
  nvec, layout   columns of a matmul and "row" or "col"
  count, iters   matrices of a CG batch and iterations of a pass

The point set and the H2 representation of a case are the plan that a program
builds once and keeps; they are made once per process and uploaded anew for
each state.  The vectors come from the seed.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from h2pack_amd import abi
from h2pack_amd import construct as C
from h2pack_amd.h2mat import H2Batch, H2MatHIP

KID = {"coulomb": C.KRNL_COULOMB, "gaussian": C.KRNL_GAUSSIAN, "matern32": C.KRNL_MATERN32,
       "rpy": C.KRNL_RPY, "rpy_periodic": C.KRNL_RPY}
DEV = "cuda:0"
# largest point set whose dense product is formed in exact()
EXACT_MAX_N = 450_000


def listed():
    return [
        # one FP64 product of the benchmark's default workload: a million
        # points of a Gaussian process, the largest matrix in use
        {"name": "gaussian 1M matvec", "op": "matvec", "kernel": "gaussian", "n": 1_000_000, "density": 10.0,
         "l": 1.0, "leaf": 300, "reltol": 1e-6, "mode": "jit", "prec": "fp64"},
        # the smallest calls: a few thousand points, where launches and
        # latency are what a solver's inner loop waits for
        {"name": "gaussian 4k matvec", "op": "matvec", "kernel": "gaussian", "n": 4000, "density": 10.0,
         "l": 1.0, "leaf": 150, "reltol": 1e-6, "mode": "jit", "prec": "fp64"},
        # stored blocks streamed from HBM, the mode of a program that applies
        # one matrix many times and has the memory
        {"name": "coulomb 80k aot matvec", "op": "matvec", "kernel": "coulomb", "n": 80_000, "density": 1.0,
         "l": 0.0, "leaf": 300, "reltol": 1e-6, "mode": "aot", "prec": "fp64"},
        # electrostatics on a large dense point set, blocks evaluated in the call
        {"name": "coulomb 200k matvec", "op": "matvec", "kernel": "coulomb", "n": 200_000, "density": 10.0,
         "l": 0.0, "leaf": 300, "reltol": 1e-6, "mode": "jit", "prec": "fp64"},
        # a serving request of the mean size, FP32-mixed: the product that
        # each iteration of its solve waits for
        {"name": "matern 105k fp32mix matvec", "op": "matvec", "kernel": "matern32", "n": 105_501, "density": 10.0,
         "l": 0.8, "leaf": 300, "reltol": 1e-6, "mode": "jit", "prec": "fp32mix"},
        # Brownian dynamics: one mobility product (3 x 3 tensor kernel)
        {"name": "rpy 20k matvec", "op": "matvec", "kernel": "rpy", "n": 20_011, "density": 0.2,
         "l": 1.0, "leaf": 200, "reltol": 1e-7, "mode": "jit", "prec": "fp64"},
        # the same mobility matrix on a block of random vectors
        {"name": "rpy 20k matmul x32", "op": "matmul", "kernel": "rpy", "n": 20_011, "density": 0.2,
         "l": 1.0, "leaf": 200, "reltol": 1e-7, "mode": "jit", "prec": "fp64", "nvec": 32, "layout": "col"},
        # the 8 right-hand sides of a serving request
        {"name": "matern 105k fp32mix matmul x8", "op": "matmul", "kernel": "matern32", "n": 105_501,
         "density": 10.0, "l": 0.8, "leaf": 300, "reltol": 1e-6, "mode": "jit", "prec": "fp32mix", "nvec": 8,
         "layout": "col"},
        # a block of vectors on stored blocks, row-major as numpy holds it
        {"name": "gaussian 17k aot matmul x64", "op": "matmul", "kernel": "gaussian", "n": 17_001, "density": 10.0,
         "l": 1.0, "leaf": 300, "reltol": 1e-6, "mode": "aot", "prec": "fp64", "nvec": 64, "layout": "row"},
        # an odd number of columns in FP64 with the blocks evaluated in the call
        {"name": "coulomb 80k matmul x20", "op": "matmul", "kernel": "coulomb", "n": 80_000, "density": 1.0,
         "l": 0.0, "leaf": 300, "reltol": 1e-6, "mode": "jit", "prec": "fp64", "nvec": 20, "layout": "row"},
        # several Gaussian-process solves advanced together, as the server does
        {"name": "matern cg x3", "op": "cg", "kernel": "matern32", "n": 24_001, "density": 10.0, "l": 1.0,
         "leaf": 300, "reltol": 1e-6, "mode": "jit", "prec": "fp64", "count": 3, "iters": 10},
        # a periodic suspension
        {"name": "rpy periodic 10k matvec", "op": "matvec", "kernel": "rpy_periodic", "n": 10_000, "density": 0.2,
         "l": 1.0 / (6.0 * math.pi), "leaf": 200, "reltol": 1e-6, "mode": "jit", "prec": "fp64"},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["matvec", "matvec", "matvec", "matmul", "matmul", "cg"])
    if op == "cg":
        return {"op": "cg", "kernel": rng.choice(["matern32", "gaussian"]), "n": _log_uniform(rng, 6000, 30_000),
                "density": 10.0, "l": round(rng.uniform(0.6, 2.0), 3), "leaf": rng.choice([150, 300]),
                "reltol": 1e-6, "mode": "jit", "prec": "fp64", "count": rng.choice([2, 3]),
                "iters": rng.randint(5, 12)}
    kernel = rng.choice(["coulomb", "coulomb", "gaussian", "gaussian", "matern32", "matern32", "rpy"])
    c = {"op": op, "kernel": kernel, "reltol": rng.choice([1e-6, 1e-6, 1e-7])}
    if kernel == "rpy":
        c.update({"n": _log_uniform(rng, 2000, 20_000), "density": rng.choice([0.03, 0.1, 0.2]), "l": 1.0,
                  "leaf": rng.choice([120, 200]), "mode": rng.choice(["jit", "jit", "aot"]), "prec": "fp64"})
    else:
        mode = rng.choice(["jit", "jit", "jit", "aot"])
        top = 100_000 if mode == "aot" else 400_000
        if op == "matmul":
            top = 30_000 if mode == "aot" else 105_000
        c.update({"n": _log_uniform(rng, 2000, top),
                  "density": rng.choice([1.0, 10.0]) if kernel == "coulomb" else 10.0,
                  "l": 0.0 if kernel == "coulomb" else round(rng.uniform(0.5, 2.0), 3),
                  "leaf": rng.choice([150, 200, 300, 400]), "mode": mode,
                  "prec": rng.choice(["fp64", "fp64", "fp32mix"])})
    if op == "matmul":
        top = 64 if c["n"] <= 30_000 else 32 if c["n"] <= 60_000 else 16
        c.update({"nvec": _log_uniform(rng, 2, top), "layout": rng.choice(["row", "col"])})
    return c


def sizes(case):
    """Points of each matrix of the case (a CG batch has matrices of different sizes)."""
    return [case["n"] - k * (case["n"] // 4) for k in range(case.get("count", 1))]


def points(kernel, n, density):
    """(3 or 4, n) points uniform in a cube; RPY: particles of radius 1 at a volume fraction."""
    rng = np.random.default_rng(20_000 + n)
    if kernel.startswith("rpy"):
        side = (n * (4.0 / 3.0) * math.pi / density) ** (1.0 / 3.0)
        return np.concatenate([rng.random((3, n)) * side, np.ones((1, n))], axis=0), side
    side = (n / density) ** (1.0 / 3.0)
    return rng.random((3, n)) * side, side


@functools.lru_cache(maxsize=24)
def representation(kernel, n, density, l, leaf, reltol):
    """The H2 representation a program builds once on the host."""
    coord, side = points(kernel, n, density)
    if kernel == "rpy_periodic":
        return C.build_periodic(coord, [0.0, 0.0, 0.0, side, side, side], l, (side, 1.9 / side, 6, 6), reltol,
                                  leaf)
    return C.build_h2(coord, KID[kernel], [] if kernel == "coulomb" else [l], reltol, leaf, BD_JIT=1,
                      pp_kind="surface" if kernel == "rpy" else "numerical", host_blocks=False)


def representations(case):
    return [representation(case["kernel"], n, case["density"], case["l"], case["leaf"], case["reltol"])
            for n in sizes(case)]


def vectors(case, seed):
    """The case's input vectors: one per matrix, (N,) or (N, nvec)."""
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    kd = 3 if case["kernel"].startswith("rpy") else 1
    out = []
    for n in sizes(case):
        if case["op"] == "matmul":
            shape = (n * kd, case["nvec"]) if case["layout"] == "row" else (case["nvec"], n * kd)
            out.append(torch.randn(shape, generator=g, dtype=torch.float64, device=DEV))
        elif case["op"] == "cg":
            out.append(torch.randn(n * kd, generator=g, dtype=torch.float64, device=DEV))
        else:
            out.append(torch.rand(n * kd, generator=g, dtype=torch.float64, device=DEV) - 0.5)
    return out


NUGGET = 1e-2     # diagonal shift of the CG solves


def prepare(case, seed):
    ins = vectors(case, seed)
    s = {"case": case, "in": ins, "out": [torch.zeros_like(v) for v in ins],
         "mats": [H2MatHIP(h, mode=case["mode"], prec=case["prec"], host_blocks=False)
                  for h in representations(case)]}
    if case["op"] == "cg":
        s["batch"] = H2Batch()
    return s


def run(s):
    case, m = s["case"], s["mats"][0]
    x, y = s["in"][0], s["out"][0]
    stream = torch.cuda.current_stream().cuda_stream
    if case["op"] == "matvec":
        m.matvec_dev(x.data_ptr(), y.data_ptr(), stream)
        return y
    if case["op"] == "matmul":
        row = case["layout"] == "row"
        ld = case["nvec"] if row else m.N
        m.matmul_dev(abi.ROW_MAJOR if row else abi.COL_MAJOR, case["nvec"], x.data_ptr(), ld, y.data_ptr(), ld,
                     stream)
        return y
    # a batch of CG solves from x = 0, a fixed number of iterations, then the
    # poll that a server makes after each tick
    k = len(s["mats"])
    for v in s["out"]:
        v.zero_()
    b = s["batch"]
    b.cg_start(s["mats"], [v.data_ptr() for v in s["in"]], [v.data_ptr() for v in s["out"]], [NUGGET] * k,
               [1e-12] * k, [1000] * k, stream)
    b.cg_step(s["mats"], case["iters"], stream)
    done, iters, relres = b.cg_poll(s["mats"], stream)
    return {"x": s["out"], "done": done, "iters": iters, "relres": relres}


def work(case):
    """Each stored entry, coordinate and vector entry once; per kernel pair the
    flops the reference counts for its kernels (matvec), or a multiply-add per
    entry, direction and column (matmul)."""
    flops = byts = 0.0
    for h in representations(case):
        kd = h.krnl_dim
        U = sum(float(u.size) for u in h.U)
        B, D = float(h.B_ptr[-1]), float(h.D_ptr[-1])
        nv = case.get("nvec", 1)
        byts += 8.0 * U + 16.0 * h.krnl_mat_size * nv + 8.0 * h.xpt_dim * h.n_point
        if case["mode"] == "aot":
            byts += (4.0 if case["prec"] == "fp32mix" else 8.0) * (B + D)
        if case["op"] == "matmul":
            diag = sum(float(d) for d in np.asarray(h.D_ptr[1:h.n_leaf_node + 1], dtype=np.float64)
                       - np.asarray(h.D_ptr[:h.n_leaf_node], dtype=np.float64))
            flops += 2.0 * nv * (2 * U + 2 * B + 2 * D - diag)
        elif case["mode"] == "aot":
            flops += 4.0 * (U + B + D)
        else:
            flops += 4.0 * U + C.KRNL_BIMV_FLOPS[KID[case["kernel"]]] * (B + D) / (kd * kd)
        if case["op"] == "cg":
            byts += 8.0 * 4 * h.krnl_mat_size
    if case["op"] == "cg":
        flops, byts = flops * (case["iters"] + 1), byts * (case["iters"] + 1)
    return {"bytes": byts, "flops": flops}


def _dense_rows(kernel, l, P, i0, i1):
    """Rows of the dense kernel matrix for points i0 .. i1 - 1 against all points, FP64."""
    d = [P[a, i0:i1, None] - P[a, None, :] for a in range(3)]
    r2 = d[0] * d[0] + d[1] * d[1] + d[2] * d[2]
    if kernel == "gaussian":
        return torch.exp(-l * r2)
    if kernel == "matern32":
        t = math.sqrt(3.0) * l * torch.sqrt(r2)
        return (1.0 + t) * torch.exp(-t)
    r = torch.sqrt(r2)
    inv = torch.where(r > 0, 1.0 / r, torch.zeros_like(r))
    if kernel == "coulomb":
        return inv
    # Rotne-Prager-Yamakawa tensor of spheres of radius 1, viscosity l
    c = 1.0 / (6.0 * math.pi * l)
    far = r > 2.0
    f0 = 0.75 * inv
    t1 = torch.where(far, f0 * (1.0 + (2.0 / 3.0) * inv * inv), 1.0 - (9.0 / 32.0) * r)
    t2 = torch.where(far, f0 * (1.0 - 2.0 * inv * inv), (3.0 / 32.0) * r)
    t1, t2 = t1 * c, t2 * c * inv * inv
    m, n = r.shape
    K = torch.empty((m, 3, n, 3), dtype=torch.float64, device=P.device)
    for a in range(3):
        for b in range(3):
            K[:, a, :, b] = t2 * d[a] * d[b] + (t1 if a == b else 0.0)
    return K.reshape(3 * m, 3 * n)


def _dense_apply(case, n, X):
    """K X for X of shape (N, k), row chunk by row chunk."""
    P = torch.from_numpy(points(case["kernel"], n, case["density"])[0]).to(DEV)
    kd = 3 if case["kernel"].startswith("rpy") else 1
    rows = max(1, min(n, int(2e8 / (n * kd * kd))))
    Y = torch.empty_like(X)
    for i in range(0, n, rows):
        j = min(n, i + rows)
        Y[kd * i:kd * j] = _dense_rows(case["kernel"], case["l"], P, i, j) @ X
    return Y


def exact(case, seed):
    """The dense kernel product in 64 bits (None for the periodic sum and for
    point sets too large for it)."""
    if case["kernel"] == "rpy_periodic" or case["n"] > EXACT_MAX_N:
        return None
    ins = vectors(case, seed)
    if case["op"] == "matvec":
        return _dense_apply(case, case["n"], ins[0][:, None])[:, 0].contiguous()
    if case["op"] == "matmul":
        if case["layout"] == "row":
            return _dense_apply(case, case["n"], ins[0])
        return _dense_apply(case, case["n"], ins[0].T.contiguous()).T.contiguous()
    xs, relres = [], []
    for n, b in zip(sizes(case), ins):
        x, r = torch.zeros_like(b), b.clone()
        p, rr = r.clone(), torch.dot(r, r)
        for _ in range(case["iters"]):
            q = _dense_apply(case, n, p[:, None])[:, 0] + NUGGET * p
            a = rr / torch.dot(p, q)
            x += a * p
            r -= a * q
            new = torch.dot(r, r)
            p = r + (new / rr) * p
            rr = new
        xs.append(x)
        relres.append(float(torch.sqrt(rr) / torch.linalg.norm(b)))
    k = len(xs)
    return {"x": xs, "done": [0] * k, "iters": [case["iters"]] * k, "relres": relres}
