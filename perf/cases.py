"""The workloads by which this framework's speed is judged, each one pass through its public entry points.

A case is a dict of plain values.  ``op`` says which path it takes:

* ``mv`` / ``mvt``: ``bsr_mv`` (plain / ``transpose=True``) with a vector that the caller keeps.  Every iteration of a
  Krylov solver or an explicit time step is one; the transposed product is what adjoint solves and least squares call.
* ``assemble``: ``bsr_set_from_triplets`` into a matrix that the caller keeps, and the block count read back, as a
  nonlinear solve does once per step.
* ``cg``: ``cg`` with a (block-)Jacobi preconditioner, run for a fixed number of iterations that ends before convergence
  (so that every correct implementation ends at the same iterate).
* ``project``: a copy of an assembled system and its Dirichlet projection (``fem.project_linear_system``), as a program
  does that keeps the unconstrained matrix for its reaction forces.
* ``fcg``: flexible CG with the learned preconditioner (three smoothing products and a 3D U-Net per iteration).
* ``train``: loss and parameter gradients of one training pair through the U-Net, what gradient accumulation calls.

Matrices: ``poisson2d`` is the bilinear 2D Poisson operator (1x1 blocks, 9 entries per row), ``elasticity`` the trilinear
hexahedral 3D elasticity operator (3x3 blocks, 27 per row), ``fv7`` the 7-point finite-volume operator with a
coefficient that varies over orders of magnitude (1x1 blocks).
"""

from __future__ import annotations

import math
import os

import numpy as np
import torch

import warp_amd as wa
from warp_amd import fem, problems, sparse
from warp_amd.optim import learned, linear

DEV = "cuda"
DTYPES = {"f32": torch.float32, "f64": torch.float64}
CHECKPOINT = os.path.join(os.path.dirname(wa.__file__), "data", "fv7_unet_128.npz")
OMEGA = 2.0 / 3.0
# (name, input channels, output channels, relu, level) of the U-Net in the order of evaluation
UNET = [("e0", 2, 16, True, 0), ("e1", 16, 32, True, 1), ("e2", 32, 64, True, 2), ("e3", 64, 64, True, 3),
        ("d2", 64, 32, True, 2), ("d1", 32, 16, True, 1), ("d0", 16, 1, False, 0)]


def listed():
    return [
        # a small 2D system: what one product costs when latency and the host bound it
        {"name": "mv-poisson2d-128", "op": "mv", "family": "poisson2d", "n": 128, "dtype": "f32"},
        # the product of a mid-sized 3D elasticity solve, larger than the memory-side cache
        {"name": "mv-elasticity-64", "op": "mv", "family": "elasticity", "n": 64, "dtype": "f32"},
        # a double-precision scalar product on an odd grid
        {"name": "mv-fv7-161-f64", "op": "mv", "family": "fv7", "n": 161, "dtype": "f64"},
        # the transposed product of an adjoint solve on an odd mesh
        {"name": "mvt-elasticity-53", "op": "mvt", "family": "elasticity", "n": 53, "dtype": "f32"},
        # assembly of a small 2D system in element order, boundary triplets dropped
        {"name": "assemble-poisson2d-128", "op": "assemble", "family": "poisson2d", "n": 128, "dtype": "f32", "order": "element"},
        # assembly of 16.8 million 3x3 triplets in no order (elements processed in any order, several per thread)
        {"name": "assemble-elasticity-64", "op": "assemble", "family": "elasticity", "n": 64, "dtype": "f32", "order": "shuffled"},
        # a small solve: launches and latency bound each iteration
        {"name": "cg-poisson2d-128", "op": "cg", "family": "poisson2d", "n": 128, "dtype": "f32", "prec": "diag", "iters": 80},
        # a block-Jacobi elasticity solve
        {"name": "cg-elasticity-64", "op": "cg", "family": "elasticity", "n": 64, "dtype": "f32", "prec": "block_diag", "iters": 40},
        # the inner solve of the mixed-precision refinement on 16.8 million unknowns
        {"name": "cg-fv7-256", "op": "cg", "family": "fv7", "n": 256, "dtype": "f32", "prec": "diag", "iters": 40},
        # boundary conditions of the elasticity system: one clamped face, one face that slides along random planes
        {"name": "project-elasticity-64", "op": "project", "family": "elasticity", "n": 64, "dtype": "f32"},
        # the learned solver at the size that its shipped network is trained for
        {"name": "fcg-fv7-128", "op": "fcg", "n": 128, "iters": 8},
        # one gradient of that network's training
        {"name": "train-fv7-128", "op": "train", "n": 128, "precision": "bf16"},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    op = rng.choice(["mv", "mv", "mvt", "assemble", "assemble", "cg", "cg", "project", "fcg", "train"])
    if op in ("fcg", "train"):
        n = rng.choice([32, 64, 96, 128])
        if op == "fcg":
            return {"op": op, "n": n, "iters": 2 * rng.randint(1, 4)}
        precision = "bf16" if n > 64 else rng.choice(["bf16", "bf16", "fp32"])
        return {"op": op, "n": n, "precision": precision}
    dtype = rng.choice(["f32", "f32", "f64"])
    if op == "assemble":
        family = rng.choice(["poisson2d", "elasticity", "elasticity", "synthetic"])
        if family == "synthetic":  # random keys, many duplicates per block: rows of 70 and more triplets
            return {"op": op, "family": family, "n": log_int(8, 40), "dtype": dtype, "order": "shuffled"}
        n = log_int(16, 700) if family == "poisson2d" else log_int(4, 64 if dtype == "f32" else 48)
        return {"op": op, "family": family, "n": n, "dtype": dtype, "order": rng.choice(["element", "shuffled"])}
    if op == "project":
        return {"op": op, "family": "elasticity", "n": log_int(6, 64 if dtype == "f32" else 48), "dtype": dtype}
    family = rng.choice(["poisson2d", "elasticity", "fv7"])
    n = {"poisson2d": log_int(16, 700), "elasticity": log_int(6, 64 if dtype == "f32" else 50),
         "fv7": log_int(16, 256 if dtype == "f32" else 180)}[family]
    if op == "cg":
        # well before convergence, where the iterate does not yet depend on rounding
        iters = max(4, min({"poisson2d": 80, "elasticity": 40, "fv7": 40}[family], int(0.6 * n)))
        prec = rng.choice(["diag", "block_diag"]) if family == "elasticity" else "diag"
        return {"op": op, "family": family, "n": n, "dtype": dtype, "prec": prec, "iters": iters}
    return {"op": op, "family": family, "n": n, "dtype": dtype}


# ---------------------------------------------------------------------------
# Inputs (from the seed alone)
# ---------------------------------------------------------------------------


def _gen(seed, k):
    return torch.Generator(device=DEV).manual_seed(1_000_003 * (seed + 1) + k)


def _compact(rows, cols, vals, nrow):
    """Offsets, columns and values of the summed triplets (duplicates summed in 64 bits, then rounded)."""
    keep = (rows >= 0) & (cols >= 0)
    rows, cols, vals = rows[keep], cols[keep], vals[keep]
    key, inv = torch.unique(rows.to(torch.int64) * nrow + cols, sorted=True, return_inverse=True)
    out = torch.zeros((key.numel(),) + tuple(vals.shape[1:]), dtype=torch.float64, device=vals.device)
    out.index_add_(0, inv, vals.to(torch.float64))
    offsets = torch.zeros(nrow + 1, dtype=torch.int64, device=vals.device)
    offsets[1:] = torch.cumsum(torch.bincount(key // nrow, minlength=nrow), 0)
    return offsets.to(torch.int32), (key % nrow).to(torch.int32), out


def _smooth_field(n, seed):
    """A smooth random field of unit deviation on n^3 cells (correlated over about 16 cells)."""
    m = max(3, n // 16 + 2)
    g = torch.randn((1, 1, m, m, m), generator=_gen(seed, 1), device=DEV, dtype=torch.float32)
    g = torch.nn.functional.interpolate(g, size=(n, n, n), mode="trilinear", align_corners=True)[0, 0]
    return (g - g.mean()) / g.std()


def _matrix(case, seed):
    """(offsets, columns, values [nnz, b, b], right-hand side, block rows, block size) of a case's operator."""
    n, dt = case["n"], DTYPES[case["dtype"]]
    if case["family"] == "poisson2d":
        rows, cols, vals, b, nrow = problems.poisson2d_q1(n, seed)
        rows, cols, vals, b = (torch.from_numpy(t).to(DEV) for t in (rows, cols, vals, b))
        off, col, val = _compact(rows, cols, vals.view(-1, 1, 1), nrow)
        return off, col, val.to(dt), b.to(dt), nrow, 1
    if case["family"] == "elasticity":
        rows, cols, vals, b, nrow = problems.elasticity3d_q1(n, 2 * seed + 1, 2 * seed + 2, device=DEV)
        off, col, val = _compact(rows, cols, vals, nrow)
        return off, col, val.to(dt), b.to(dt), nrow, 3
    k = torch.exp(2.3 * _smooth_field(n, seed))
    off, col, val = problems.fv7_poisson(k)
    b = torch.randn(n**3, generator=_gen(seed, 2), device=DEV, dtype=torch.float32) / (n * n)
    return off, col, val.to(dt).view(-1, 1, 1), b.to(dt), n**3, 1


def _bsr(case, off, col, val, nrow, bs):
    scalar = wa.float64 if case["dtype"] == "f64" else wa.float32
    A = sparse.bsr_zeros(nrow, nrow, scalar if bs == 1 else wa.matrix(shape=(bs, bs), dtype=scalar), device=DEV)
    A.offsets, A.columns, A.values = off, col, (val.reshape(-1) if bs == 1 else val).contiguous()
    A.nnz = int(col.numel())
    return A


def _vector(case, seed, nrow, bs):
    x = torch.randn((nrow, bs), generator=_gen(seed, 3), device=DEV, dtype=torch.float32).to(DTYPES[case["dtype"]])
    return x.reshape(-1).contiguous() if bs == 1 else x


def _triplets(case, seed):
    """(rows, columns, values, block rows, block size) of an assembly."""
    n, dt = case["n"], DTYPES[case["dtype"]]
    if case["family"] == "synthetic":
        u = min(9 * n**3, (3 * n + 1) ** 3)
        rows, cols, vals, nrow = problems.synthetic_triplets(n, 8 * u, u, seed, device=DEV)
        return rows, cols, vals.to(dt), nrow, 3
    if case["family"] == "elasticity":
        if case["order"] == "shuffled":
            rows, cols, vals, nrow = problems.elasticity_triplets_shuffled(n, 2 * seed + 1, 2 * seed + 2, device=DEV)
        else:
            rows, cols, vals, _, nrow = problems.elasticity3d_q1(n, 2 * seed + 1, 2 * seed + 2, device=DEV)
        return rows, cols, vals.to(dt), nrow, 3
    rows, cols, vals, _, nrow = problems.poisson2d_q1(n, seed)
    rows, cols, vals = (torch.from_numpy(np.ascontiguousarray(t)).to(DEV) for t in (rows, cols, vals))
    # a coefficient per element, so that no two systems are alike
    vals = vals * torch.exp(torch.randn(n * n, generator=_gen(seed, 4), device=DEV)).repeat_interleave(16)
    if case["order"] == "shuffled":
        perm = torch.randperm(rows.numel(), generator=_gen(seed, 5), device=DEV)
        rows, cols, vals = rows[perm], cols[perm], vals[perm]
    return rows.contiguous(), cols.contiguous(), vals.to(dt).contiguous(), nrow, 1


def _constraints(case, seed, nrow):
    """(constrained nodes, projector blocks, fixed values per node): the x = 0 face clamped, the y = 0 face sliding on
    random planes."""
    n, dt = case["n"], DTYPES[case["dtype"]]
    p = n + 1
    node = torch.arange(nrow, device=DEV)
    clamped = node % p == 0
    slides = ((node // p) % p == 0) & ~clamped
    idx = torch.nonzero(clamped | slides).reshape(-1)
    normal = torch.randn((idx.numel(), 3), generator=_gen(seed, 6), device=DEV, dtype=torch.float64)
    normal = normal / normal.norm(dim=1, keepdim=True)
    blocks = normal[:, :, None] * normal[:, None, :]
    blocks[clamped[idx]] = torch.eye(3, dtype=torch.float64, device=DEV)
    fixed = torch.randn((nrow, 3), generator=_gen(seed, 7), device=DEV, dtype=torch.float64)
    return idx, blocks.to(dt).contiguous(), fixed.to(dt)


def _fv7_system(case, seed):
    """(offsets, columns, values, b, log k) of the operator family that the network is trained on."""
    off, col, val, b, k = problems.fv7_problem(case["n"], 1.5, 8.0, seed, seed + 1_000_003, device=DEV)
    return off, col, val, b, torch.log(k).reshape(-1)


def _pair(case, seed, off, col, val):
    """A training pair A e = r, both scaled to rms(r) = 1."""
    n = case["n"]
    e = _smooth_field(n, seed).reshape(-1).to(torch.float64)
    e = e + 0.1 * torch.randn(n**3, generator=_gen(seed, 8), device=DEV, dtype=torch.float32)
    r = _product(off, col, val.to(torch.float64).view(-1, 1, 1), e.view(-1, 1)).reshape(-1)
    s = r.pow(2).mean().sqrt()
    return (r / s).to(torch.float32), (e / s).to(torch.float32)


# ---------------------------------------------------------------------------
# Preparation and one pass
# ---------------------------------------------------------------------------


def prepare(case, seed):
    op = case["op"]
    if op in ("mv", "mvt"):
        off, col, val, _, nrow, bs = _matrix(case, seed)
        x = _vector(case, seed, nrow, bs)
        return {"op": op, "A": _bsr(case, off, col, val, nrow, bs), "x": x, "y": torch.zeros_like(x)}
    if op == "assemble":
        rows, cols, vals, nrow, bs = _triplets(case, seed)
        scalar = wa.float64 if case["dtype"] == "f64" else wa.float32
        A = sparse.bsr_zeros(nrow, nrow, scalar if bs == 1 else wa.matrix(shape=(bs, bs), dtype=scalar), device=DEV)
        return {"op": op, "A": A, "rows": rows, "cols": cols, "vals": vals}
    if op == "cg":
        off, col, val, b, nrow, bs = _matrix(case, seed)
        A = _bsr(case, off, col, val, nrow, bs)
        return {"op": op, "A": A, "b": b, "x": torch.zeros_like(b), "M": linear.preconditioner(A, case["prec"]),
                "iters": case["iters"]}
    if op == "project":
        off, col, val, b, nrow, bs = _matrix(case, seed)
        idx, blocks, fixed = _constraints(case, seed, nrow)
        poff = torch.zeros(nrow + 1, dtype=torch.int64, device=DEV)
        poff[idx + 1] = 1
        P = _bsr(case, torch.cumsum(poff, 0).to(torch.int32), idx.to(torch.int32), blocks, nrow, bs)
        return {"op": op, "A": _bsr(case, off, col, val, nrow, bs), "b": b, "P": P, "fixed": fixed}
    system = learned.FV7System(case["n"], 1.5, 8.0, seed, DEV)
    if op == "fcg":
        net, _ = learned.load_checkpoint(CHECKPOINT, case["n"], DEV)
        return {"op": op, "fcg": learned.LearnedFCG(system, net, smooth_steps=1, omega=OMEGA),
                "x": torch.zeros(case["n"] ** 3, dtype=torch.float64, device=DEV), "iters": case["iters"]}
    net = learned.UNet(case["n"], DEV, seed=seed % 997)
    A = system.A
    r, e = _pair(case, seed, A.offsets, A.columns, A.values)
    return {"op": op, "trainer": learned.EnergyTrainer(net, smooth_steps=1, omega=OMEGA, precision=case["precision"]),
            "system": system, "r": r, "e": e}


def run(state):
    op = state["op"]
    if op in ("mv", "mvt"):
        return sparse.bsr_mv(state["A"], state["x"], state["y"], transpose=op == "mvt")
    if op == "assemble":
        A = state["A"]
        sparse.bsr_set_from_triplets(A, state["rows"], state["cols"], state["vals"])
        nnz = A.nnz_sync()
        return {"offsets": A.offsets, "columns": A.columns[:nnz], "values": A.values[:nnz]}
    if op == "cg":
        state["x"].zero_()
        it, err, _ = linear.cg(state["A"], state["b"], state["x"], tol=1e-10, atol=0.0, maxiter=state["iters"], M=state["M"])
        return {"x": state["x"], "iterations": it, "residual": err}
    if op == "project":
        A, b = sparse.bsr_copy(state["A"]), state["b"].clone()
        fem.project_linear_system(A, b, state["P"], state["fixed"], normalize_projector=False)
        nnz = A.nnz_sync()
        return {"offsets": A.offsets, "columns": A.columns[:nnz], "values": A.values[:nnz], "b": b}
    if op == "fcg":
        state["x"].zero_()
        state["fcg"].solve(state["x"], tol=1e-8, maxiter=state["iters"], use_graph=False, fallback=False)
        return state["x"]
    loss = state["trainer"].gradient(state["system"], state["r"], state["e"])
    return {"loss": loss, **state["trainer"].net.grads}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------


def _size(case):
    """(block rows, blocks, block size) of a case's operator."""
    n = case["n"]
    if case["family"] == "poisson2d":
        return (n - 1) ** 2, (3 * (n - 1) - 2) ** 2, 1
    if case["family"] == "elasticity":
        return (n + 1) ** 3, (3 * n + 1) ** 3, 3
    return n**3, 7 * n**3 - 6 * n**2, 1


def work(case):
    op, n = case["op"], case["n"]
    if op in ("fcg", "train"):
        N, nnz = n**3, 7 * n**3 - 6 * n**2
        net_flops = sum(2 * 27 * ci * co * (n >> lvl) ** 3 for _, ci, co, _, lvl in UNET)
        size = 4 if case.get("precision") == "fp32" else 2
        # each activation written once and read once by each of its readers
        net_bytes = sum(size * (n >> lvl) ** 3 * (ci + co) for _, ci, co, _, lvl in UNET)
        if op == "fcg":  # three dependent products, and x, r, p, q read and written in 64 bits
            return {"bytes": case["iters"] * (3 * (8 * nnz + 4 * N) + 8 * 8 * N + net_bytes), "flops": case["iters"] * (net_flops + 6 * nnz)}
        # forward, input gradients, weight gradients; four products with the matrix
        return {"bytes": 4 * (8 * nnz + 4 * N) + 3 * net_bytes, "flops": 3 * net_flops + 8 * nnz}
    s = 8 if case["dtype"] == "f64" else 4
    if op == "assemble":
        if case["family"] == "synthetic":
            u = min(9 * n**3, (3 * n + 1) ** 3)
            nrow, blocks, triplets, bs = (n + 1) ** 3, u, 8 * u, 3
        elif case["family"] == "poisson2d":
            nrow, blocks, bs = _size(case)
            triplets = 16 * n**2
        else:
            nrow, blocks, bs = _size(case)
            triplets = 64 * n**3
        return {"bytes": triplets * (8 + bs * bs * s) + blocks * (4 + bs * bs * s) + 4 * (nrow + 1), "flops": triplets * bs * bs}
    nrow, nnz, bs = _size(case)
    matrix = nnz * (4 + bs * bs * s) + 4 * (nrow + 1)
    vec = nrow * bs * s
    if op in ("mv", "mvt"):
        return {"bytes": matrix + 2 * vec, "flops": 2 * nnz * bs * bs}
    if op == "cg":  # per iteration: the matrix, x, r and p read and written, Ap, the preconditioner
        prec = vec * (bs if case["prec"] == "block_diag" else 1)
        return {"bytes": case["iters"] * (matrix + 8 * vec + prec), "flops": case["iters"] * (2 * nnz * bs * bs + 10 * nrow * bs)}
    return {"bytes": 2 * matrix + 3 * vec, "flops": 4 * nnz * bs**3}  # project: the system read, the projected one written


def tolerance(case):
    """About four times what two summation orders, or one of them and 64 bits, were seen to differ by."""
    op = case["op"]
    if op in ("fcg", "train"):
        if case.get("precision") == "fp32":
            return {"rel": 1e-4, "max": 1e-2}
        return {"rel": 1e-2, "max": 0.3} if op == "fcg" else {"rel": 3e-2, "max": 0.5}
    f64 = case["dtype"] == "f64"
    if op == "cg":
        return {"rel": 1e-11, "max": 1e-9} if f64 else {"rel": 2e-5, "max": 2e-3}
    return {"rel": 2e-15, "max": 1e-13} if f64 else {"rel": 5e-7, "max": 2e-5}


# ---------------------------------------------------------------------------
# The same results in 64 bits, in plain torch
# ---------------------------------------------------------------------------


def _rows_of(off):
    return torch.repeat_interleave(torch.arange(off.numel() - 1, device=off.device), (off[1:] - off[:-1]).long())


def _product(off, col, val, x, rows=None):
    """A x for 64-bit blocks [nnz, b, b] and x [nrow, b]."""
    rows = _rows_of(off) if rows is None else rows
    y = torch.zeros((off.numel() - 1, val.shape[1]), dtype=torch.float64, device=val.device)
    part = val[:, 0, :] * x[col.long()] if val.shape[1] == 1 else (val * x[col.long()][:, None, :]).sum(2)
    return y.index_add(0, rows, part)


def _exact_cg(case, seed):
    off, col, val, b, nrow, bs = _matrix(case, seed)
    val, b = val.to(torch.float64), b.to(torch.float64).view(nrow, bs)
    rows = _rows_of(off)
    on = rows == col
    diag = val[on]
    if case["prec"] == "block_diag" and bs > 1:
        inv = torch.linalg.inv(diag)
        apply = lambda r: (inv * r[:, None, :]).sum(2)  # noqa: E731
    else:
        inv = 1.0 / torch.diagonal(diag, dim1=1, dim2=2)
        apply = lambda r: inv * r  # noqa: E731
    x = torch.zeros_like(b)
    r = b.clone()
    z = apply(r)
    p, rz = z, (r * z).sum()
    for _ in range(case["iters"]):
        q = _product(off, col, val, p, rows)
        alpha = rz / (p * q).sum()
        x = x + alpha * p
        r = r - alpha * q
        z = apply(r)
        rz, old = (r * z).sum(), rz
        p = z + (rz / old) * p
    shape = (nrow,) if bs == 1 else (nrow, bs)
    return {"x": x.view(shape), "iterations": None, "residual": float(r.norm())}


def _exact_assemble(case, seed):
    rows, cols, vals, nrow, bs = _triplets(case, seed)
    vals = vals.view(-1, bs, bs)
    keep = (rows >= 0) & (rows < nrow) & (cols >= 0) & (cols < nrow) & (vals != 0).flatten(1).any(1)
    off, col, val = _compact(rows[keep], cols[keep], vals[keep], nrow)
    return {"offsets": None, "columns": None, "values": val.reshape(-1) if bs == 1 else val}


def _exact_project(case, seed):
    off, col, val, b, nrow, bs = _matrix(case, seed)
    idx, blocks, fixed = _constraints(case, seed, nrow)
    P = torch.zeros((nrow, bs, bs), dtype=torch.float64, device=DEV)
    P[idx] = blocks.to(torch.float64)
    val, b, v = val.to(torch.float64), b.to(torch.float64), fixed.to(torch.float64)
    Q = torch.eye(bs, dtype=torch.float64, device=DEV) - P
    rows, c = _rows_of(off), col.long()
    left = (Q[rows][:, :, :, None] * val[:, None, :, :]).sum(2)
    out = (left[:, :, :, None] * Q[c][:, None, :, :]).sum(2)
    out = out + torch.where((rows == c)[:, None, None], P[rows], torch.zeros_like(out))
    pv = (P * v[:, None, :]).sum(2)
    rest = b - _product(off, col, val, pv, rows)
    rhs = (Q * rest[:, None, :]).sum(2) + pv
    return {"offsets": None, "columns": None, "values": out, "b": rhs}


def _conv(x, w, bias, relu):
    """3x3x3 convolution of x [z, y, x, channel], zero padding; w [tap, in, out], taps dz slowest."""
    n = x.shape[0]
    y = bias.expand(n, n, n, -1)
    xp = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    for t in range(27):
        dz, dy, dx = t // 9, (t // 3) % 3, t % 3
        y = y + xp[dz:dz + n, dy:dy + n, dx:dx + n].reshape(n**3, -1).matmul(w[t]).view(n, n, n, -1)
    return torch.relu(y) if relu else y


def _unet(p, x):
    pool = lambda a: a.view(a.shape[0] // 2, 2, a.shape[0] // 2, 2, a.shape[0] // 2, 2, -1).mean(dim=(1, 3, 5))  # noqa: E731
    up = lambda a: a.repeat_interleave(2, 0).repeat_interleave(2, 1).repeat_interleave(2, 2)  # noqa: E731
    conv = {name: (lambda v, name=name, relu=relu: _conv(v, p[name + ".W"], p[name + ".b"], relu)) for name, _, _, relu, _ in UNET}
    a0 = conv["e0"](x)
    a1 = conv["e1"](pool(a0))
    a2 = conv["e2"](pool(a1))
    a3 = conv["e3"](pool(a2))
    b2 = conv["d2"](up(a3) + a2)
    b1 = conv["d1"](up(b2) + a1)
    return conv["d0"](up(b1) + a0).reshape(-1)


def _composite(case, seed, p):
    """(matrix product, preconditioner z = M(r), b) of the learned solver's operator with the network's parameters p."""
    n = case["n"]
    off, col, val, b, logk = _fv7_system(case, seed)
    val = val.to(torch.float64).view(-1, 1, 1)
    rows = _rows_of(off)
    A = lambda v: _product(off, col, val, v.view(-1, 1), rows).reshape(-1)  # noqa: E731
    dinv = 1.0 / val[rows == col].reshape(-1)
    dmean = (1.0 / dinv).mean()
    feature = ((logk - logk.mean()) / logk.std().clamp_min(1e-12)).to(torch.float64)

    def precondition(r):
        z = OMEGA * dinv * r
        r1 = r - A(z)
        s = r1.pow(2).mean().sqrt()
        z = z + s / dmean * _unet(p, torch.stack([r1 / s, feature], 1).view(n, n, n, 2))
        return z + OMEGA * dinv * (r - A(z))

    return A, precondition, b.to(torch.float64), (off, col, val)


def _exact_fcg(case, seed):
    with np.load(CHECKPOINT, allow_pickle=False) as f:
        p = {k + part: torch.from_numpy(f[k + part]).to(DEV).to(torch.float64) for k, *_ in UNET for part in (".W", ".b")}
    A, M, b, _ = _composite(case, seed, p)
    x, r = torch.zeros_like(b), b.clone()
    d = q = torch.zeros_like(b)
    dq = 1.0
    for _ in range(case["iters"]):
        z = M(r)
        d = z - ((z * q).sum() / dq) * d
        q = A(d)
        dq = (d * q).sum()
        alpha = (d * r).sum() / dq
        x = x + alpha * d
        r = r - alpha * q
    return x


def _exact_train(case, seed):
    p = {}
    rng = np.random.default_rng(seed % 997)  # the initial weights: He-normal, drawn layer by layer
    for name, ci, co, relu, _ in UNET:
        w = (rng.standard_normal((27, ci, co)) * math.sqrt((2.0 if relu else 1.0) / (27 * ci))).astype(np.float32)
        p[name + ".W"] = torch.from_numpy(w).to(DEV).to(torch.float64).requires_grad_()
        p[name + ".b"] = torch.zeros(co, dtype=torch.float64, device=DEV, requires_grad=True)
    A, M, _, (off, col, val) = _composite(case, seed, p)
    r, e = (t.to(torch.float64) for t in _pair(case, seed, off, col, val.reshape(-1)))
    z = M(r)
    loss = 1.0 - (r * z).sum() ** 2 / ((r * e).sum() * (z * A(z)).sum())
    grads = torch.autograd.grad(loss, list(p.values()))
    return {"loss": loss.detach().reshape(1), **dict(zip(p, grads))}


def exact(case, seed):
    op = case["op"]
    if op in ("mv", "mvt"):
        off, col, val, _, nrow, bs = _matrix(case, seed)
        x = _vector(case, seed, nrow, bs).to(torch.float64).view(nrow, bs)
        val = val.to(torch.float64)
        if op == "mvt":
            rows = _rows_of(off)
            part = (val * x[rows][:, :, None]).sum(1)
            y = torch.zeros_like(x).index_add(0, col.long(), part)
        else:
            y = _product(off, col, val, x)
        return y.reshape(-1) if bs == 1 else y
    return {"assemble": _exact_assemble, "cg": _exact_cg, "project": _exact_project, "fcg": _exact_fcg,
            "train": _exact_train}[op](case, seed)
