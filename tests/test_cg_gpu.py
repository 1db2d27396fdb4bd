"""GPU conjugate gradient: reference solver scenarios and parity with the oracle.

Scenarios of the reference suite (test_linear_solvers.py:15-126, 129-253)
check err <= atol and the true residual (<= 2 atol in fp64, <= 32 atol in
fp32).  On FEM systems the native solver is compared with the oracle CG
that uses the same FP64-dot policy: same iteration count (checks happen at
the same multiples of check_every) and solutions within 1e-5 relative.
"""

from __future__ import annotations

import math

import numpy as np
import pytest
import torch

import warp_amd as wa
from warp_amd import problems, sparse
from warp_amd.optim import linear

pytestmark = pytest.mark.gpu


def _spd(n, seed, dtype, device):
    rng = np.random.default_rng(seed)
    C = rng.uniform(-100, 100, (n, n))
    f = rng.uniform(-100, 100, n)
    return torch.tensor(C @ C.T, dtype=dtype, device=device), torch.tensor(C @ f, dtype=dtype, device=device)


def _solve_with_route(A, b, x, **kw):
    """(results of cg, the plan's column window, finished workgroups of a one-launch solve)."""
    from warp_amd import _native

    solver = linear.cg(A, b, x, run=False, **kw)
    res = solver()
    off = [_native.lib().warp_amd_cg_state_offset(k) for k in (3, 4)]
    window, finished = (int(solver._ws[o:o + 4].view(torch.int32)) for o in off)
    return res, window, finished


def _check_linear_solve(A, b, **kwargs):
    x = torch.zeros_like(b)
    niter, err, atol = linear.cg(A, b, x, use_cuda_graph=True, **kwargs)
    assert err <= atol
    # device-side convergence (check_every = 0) returns device tensors
    x.zero_()
    niter0, err0, atol0 = linear.cg(A, b, x, check_every=0, **kwargs)
    assert math.sqrt(float(err0.item())) <= math.sqrt(float(atol0.item()))
    # warm start
    niter_warm, err, atol = linear.cg(A, b, x, use_cuda_graph=False, **kwargs)
    assert err <= atol
    An = A.cpu().numpy().astype(np.float64) if isinstance(A, torch.Tensor) else None
    if An is not None:
        res = np.linalg.norm(An @ x.cpu().numpy().astype(np.float64) - b.cpu().numpy())
        assert res <= (2.0 if b.dtype == torch.float64 else 32.0) * atol


def test_cg_reference_dense_scenarios(device):
    """test_cg (test_linear_solvers.py:112-126), generic operator route."""
    A, b = _spd(64, 123, torch.float64, device)
    M = linear.preconditioner(A, "diag")
    _check_linear_solve(A, b, maxiter=1000)
    _check_linear_solve(A, b, M=M, maxiter=1000)
    A, b = _spd(16, 321, torch.float32, device)
    M = linear.preconditioner(A, "diag")
    _check_linear_solve(A, b, maxiter=1000)
    _check_linear_solve(A, b, M=M, maxiter=1000)
    rng = np.random.default_rng(321)
    A = torch.eye(5, dtype=torch.float32, device=device)
    b = torch.tensor(rng.uniform(-1, 1, 5), dtype=torch.float32, device=device)
    _check_linear_solve(A, b, maxiter=30)


def test_cg_restart_callbacks(device):
    """test_conjugate_solver_restart (test_linear_solvers.py:129-172) for cg."""
    rng = np.random.default_rng(2027)
    C = rng.standard_normal((12, 12))
    A_np = C.T @ C + 4.0 * np.eye(12)
    b_np = rng.standard_normal(12)
    A = torch.tensor(A_np, device=device)
    b = torch.tensor(b_np, device=device)
    M = linear.preconditioner(A, "diag")
    for prec in (None, M):
        its = []
        x = torch.zeros_like(b)
        niter, err, atol = linear.cg(A, b, x, tol=1e-10, maxiter=120, M=prec, callback=lambda i, r, t: its.append(i),
                                     check_every=1, restart=3)
        assert err <= atol and niter % 3 == 0
        assert its[0] == 0 and its[-1] == niter and all(i % 3 == 0 for i in its)
        assert np.linalg.norm(A_np @ x.cpu().numpy() - b_np) <= atol


def _restart_drift_system(batch_count):
    """_make_cg_restart_drift_system (test_linear_solvers.py:175-201): a
    130-dof mass + spring chain with every 17th dof fixed (identity row and
    column), stacked batch_count times block-diagonally; x0 = 0.1 N(0,1)
    (seed 7301) and b = mass x0, both zero on the fixed dofs."""
    dof_count = 130
    chain_count = dof_count - 1
    edge_count = chain_count - 1
    mass = 3.0 / chain_count
    w = 0.18**2 / (3.0 / edge_count)
    A1 = mass * np.eye(dof_count)
    e = np.arange(edge_count)
    np.add.at(A1, (e, e), w)
    np.add.at(A1, (e + 1, e + 1), w)
    A1[e, e + 1] -= w
    A1[e + 1, e] -= w
    fixed = np.arange(0, chain_count, 17)
    A1[fixed, :] = 0.0
    A1[:, fixed] = 0.0
    A1[fixed, fixed] = 1.0
    A = np.kron(np.eye(batch_count), A1).astype(np.float32)
    rng = np.random.default_rng(7301)
    x0 = (0.1 * rng.standard_normal((batch_count, dof_count))).astype(np.float32)
    b = (mass * x0).astype(np.float32)
    x0[:, fixed] = 0.0
    b[:, fixed] = 0.0
    return A, b.reshape(-1), x0.reshape(-1), dof_count


@pytest.mark.parametrize("batch_count", [1, 3])
def test_cg_restart_float32_drift(device, batch_count):
    """test_cg_restart_float32_drift (test_linear_solvers.py:204-253): FP32 CG
    restarted every 32 iterations, checked every 32, graph-replayed, to
    tol 1e-6; unpreconditioned and Jacobi.  Every subproblem's FP64 true
    residual must reach tol |b_i| (restarts recompute r = b - A x, so the
    recurrence's drift cannot stop the solve short)."""
    interval, tol = 32, 1.0e-6
    A_np, b_np, x0_np, ndof = _restart_drift_system(batch_count)
    A = torch.tensor(A_np, device=device)
    b = torch.tensor(b_np, device=device)
    M = linear.preconditioner(A, "diag")
    offs = None if batch_count == 1 else _batch_offsets([ndof] * batch_count, device)
    op = linear.aslinearoperator(A, batch_offsets=offs)
    for name, prec in (("none", None), ("Jacobi", M)):
        x = torch.tensor(x0_np, device=device)
        niter, err, atol = linear.cg(op, b, x, tol=tol, atol=0.0, maxiter=512, M=prec, check_every=interval,
                                     use_cuda_graph=True, restart=interval)
        err_t, atol_t = torch.as_tensor(err), torch.as_tensor(atol)
        assert bool((err_t <= atol_t).all()), (name, err, atol)
        assert niter % interval == 0 and niter <= 512, (name, niter)
        xn = x.cpu().numpy().astype(np.float64)
        for k in range(batch_count):
            sl = slice(k * ndof, (k + 1) * ndof)
            res = A_np[sl, sl].astype(np.float64) @ xn[sl] - b_np[sl].astype(np.float64)
            target = tol * np.linalg.norm(b_np[sl].astype(np.float64))
            assert np.linalg.norm(res) <= target, f"{name} batch {k}: {np.linalg.norm(res):.3e} > {target:.3e}"


def _lanes(A):
    from warp_amd import _native

    br, bc = A.block_shape
    return _native.lib().warp_amd_bsr_mv_lanes(A.nrow, br, bc, int(A.nnz))


def _bsr_from(device, nn, rows, cols, vals, prune=True):
    block = wa.mat33 if vals.ndim == 3 else wa.float32
    A = sparse.bsr_zeros(nn, nn, block, device=device)
    sparse.bsr_set_from_triplets(A, rows.to(device), cols.to(device), vals.to(device), prune_numerical_zeros=prune)
    A.nnz_sync()
    return A


@pytest.mark.parametrize("n", [32, 128])
def test_cg_poisson_vs_oracle(device, oracle_mod, n):
    """2D Q1 Poisson, Jacobi CG, tol 1e-6, maxiter 2000 (the CPU-runnable workload at n=128)."""
    rows, cols, vals, b, nd = problems.poisson2d_q1(n, 0)
    A = _bsr_from(device, nd, torch.from_numpy(rows), torch.from_numpy(cols), torch.from_numpy(vals))
    M = linear.preconditioner(A, "diag")
    bt = torch.from_numpy(b).to(device)
    x = torch.zeros_like(bt)
    its = []
    niter, err, atol = linear.cg(A, bt, x, tol=1e-6, maxiter=2000, M=M, callback=lambda i, r, t: its.append((i, r)))
    o = oracle_mod.bsr_from_triplets(nd, nd, rows, cols, vals)
    inv = oracle_mod.inverse_diag(oracle_mod.bsr_get_diag(o["offsets"], o["columns"], o["values"]))
    G = _lanes(A)
    # oracle in the kernels' SpMV order: same trajectory up to FP64 dot rounding
    xo, it_o, err_o, atol_o, hist = oracle_mod.cg(o["offsets"], o["columns"], o["values"], b, np.zeros(nd), tol=1e-6,
                                                 maxiter=2000, prec_kind=oracle_mod.PREC_DIAG, prec=inv, group=G)
    # oracle in the reference row order
    xr, it_r, err_r, _, _ = oracle_mod.cg(o["offsets"], o["columns"], o["values"], b, np.zeros(nd), tol=1e-6,
                                         maxiter=2000, prec_kind=oracle_mod.PREC_DIAG, prec=inv)
    print(f"[cg poisson n={n}] gpu iters {niter} err {err:.3e} | oracle iters {it_o} err {err_o:.3e} "
          f"| reference-order iters {it_r} | atol {atol:.3e}")
    assert err <= atol
    assert atol == pytest.approx(atol_o, rel=1e-12)
    assert niter == it_o
    xg = x.cpu().numpy()
    assert np.linalg.norm(xg - xo) <= 1e-5 * np.linalg.norm(xo)
    assert abs(niter - it_r) <= 10
    # FP64 true residual of the FP32 solution; error vs the FP64 direct solve matches the oracle's
    import scipy.sparse as sp
    import scipy.sparse.linalg as spl

    A64 = sp.csr_matrix((o["values"].astype(np.float64), o["columns"], o["offsets"]), shape=(nd, nd))
    assert np.linalg.norm(b - A64 @ xg.astype(np.float64)) <= 32 * atol
    xs = spl.spsolve(A64.tocsc(), b.astype(np.float64))
    eg = np.linalg.norm(xg - xs) / np.linalg.norm(xs)
    er = np.linalg.norm(xr - xs) / np.linalg.norm(xs)
    print(f"[cg poisson n={n}] rel. error vs FP64 direct: gpu {eg:.3e}, reference-order oracle {er:.3e}")
    assert eg <= 1.05 * er + 1e-6
    assert its[0][0] == 0 and its[-1][0] == niter


@pytest.mark.parametrize("ptype", ["diag", "block_diag", "id"])
def test_cg_elasticity_vs_oracle(device, oracle_mod, ptype):
    n = 8
    rows, cols, vals, b, nn = problems.elasticity3d_q1(n, device="cpu")
    A = _bsr_from(device, nn, rows, cols, vals, prune=False)
    M = linear.preconditioner(A, ptype)
    bt = b.to(device)
    x = torch.zeros_like(bt)
    niter, err, atol = linear.cg(A, bt, x, tol=1e-6, atol=0.0, maxiter=5000, M=M)
    o = oracle_mod.bsr_from_triplets(nn, nn, rows.numpy(), cols.numpy(), vals.numpy(), prune=False)
    if ptype == "id":
        pk, pd = oracle_mod.PREC_NONE, None
    elif ptype == "diag":
        pk, pd = oracle_mod.PREC_DIAG, M._prec_data.cpu().numpy()
    else:
        pk, pd = oracle_mod.PREC_BLOCK, M._prec_data.cpu().numpy()
    xo, it_o, err_o, atol_o, _ = oracle_mod.cg(o["offsets"], o["columns"], o["values"], b.numpy(), np.zeros(3 * nn),
                                              tol=1e-6, atol=0.0, maxiter=5000, prec_kind=pk, prec=pd, group=_lanes(A))
    print(f"[cg elasticity {ptype}] gpu iters {niter} err {err:.3e} | oracle iters {it_o} err {err_o:.3e}")
    assert err <= atol
    assert niter == it_o
    import scipy.sparse as sp
    import scipy.sparse.linalg as spl

    A64 = sp.bsr_matrix((o["values"].astype(np.float64), o["columns"], o["offsets"]), shape=(3 * nn, 3 * nn)).tocsr()
    xs = spl.spsolve(A64.tocsc(), b.numpy().astype(np.float64).reshape(-1))
    xg = x.cpu().numpy().reshape(-1).astype(np.float64)
    rel64 = np.linalg.norm(xg - xs) / np.linalg.norm(xs)
    print(f"[cg elasticity {ptype}] rel. error vs FP64 direct solve = {rel64:.3e}")
    assert np.linalg.norm(b.numpy().reshape(-1) - A64 @ xg) <= 32 * atol
    assert np.linalg.norm(xg - xo) <= 1e-5 * np.linalg.norm(xo)


def test_cg_native_check_every_zero_and_restart(device, oracle_mod):
    rows, cols, vals, b, nd = problems.poisson2d_q1(24, 0)
    A = _bsr_from(device, nd, torch.from_numpy(rows), torch.from_numpy(cols), torch.from_numpy(vals))
    M = linear.preconditioner(A, "diag")
    bt = torch.from_numpy(b).to(device)
    x = torch.zeros_like(bt)
    it, rr, at = linear.cg(A, bt, x, tol=1e-6, atol=0.0, maxiter=500, M=M, check_every=0)
    assert isinstance(it, torch.Tensor)
    assert float(rr.item()) <= float(at.item())
    x1 = torch.zeros_like(bt)
    n1, e1, a1 = linear.cg(A, bt, x1, tol=1e-6, atol=0.0, maxiter=500, M=M, check_every=1, callback=lambda *a: None)
    # device-side convergence stops at the first converged iteration, like check_every=1 (general
    # kernels both, by the callback)
    assert int(it.item()) == n1
    np.testing.assert_array_equal(x.cpu().numpy(), x1.cpu().numpy())
    # the one-launch solve sums its dot products in another order: the same iterations, and a solution within
    # the 1e-5 that solves in the kernels' own order are held to against the oracle
    x3 = torch.zeros_like(bt)
    (n3, e3, a3), _, finished = _solve_with_route(A, bt, x3, tol=1e-6, atol=0.0, maxiter=500, M=M, check_every=1)
    assert finished > 0 and n3 == n1 and e3 <= a3
    assert float((x3 - x1).norm()) <= 1e-5 * float(x1.norm())
    # restart: true residual at the cycle boundary
    x2 = torch.zeros_like(bt)
    n2, e2, a2 = linear.cg(A, bt, x2, tol=1e-6, atol=0.0, maxiter=512, M=M, check_every=32, restart=32)
    assert n2 % 32 == 0 and e2 <= a2
    o = oracle_mod.bsr_from_triplets(nd, nd, rows, cols, vals)
    import scipy.sparse as sp

    A64 = sp.csr_matrix((o["values"].astype(np.float64), o["columns"], o["offsets"]), shape=(nd, nd))
    assert np.linalg.norm(b - A64 @ x2.cpu().numpy()) <= 2 * a2


def test_cg_functor_reuse(device):
    rows, cols, vals, b, nd = problems.poisson2d_q1(16, 0)
    A = _bsr_from(device, nd, torch.from_numpy(rows), torch.from_numpy(cols), torch.from_numpy(vals))
    bt = torch.from_numpy(b).to(device)
    x = torch.zeros_like(bt)
    solver = linear.cg(A, bt, x, tol=1e-6, run=False)
    n1, e1, a1 = solver()
    x2 = torch.zeros_like(bt)
    n2, e2, a2 = solver(b=bt, x=x2)
    assert n1 == n2 and e1 == e2
    np.testing.assert_array_equal(x.cpu().numpy(), x2.cpu().numpy())
    with pytest.raises(ValueError, match="Incompatible b.shape"):
        solver(b=torch.zeros(nd + 1, device=device))


def test_cg_zero_rhs_and_identity(device):
    """b = 0 converges before the first iteration with x = 0; the identity
    converges in one iteration (textbook special cases)."""
    n = 50
    idx = torch.arange(n, dtype=torch.int32)
    A = _bsr_from(device, n, idx, idx, torch.ones(n))
    b = torch.zeros(n, device=device)
    x = torch.zeros(n, device=device)
    it, err, atol = linear.cg(A, b, x, tol=1e-6, maxiter=100)
    assert it == 0 and err == 0.0 and torch.count_nonzero(x) == 0
    b = torch.randn(n, device=device)
    it, err, atol = linear.cg(A, b, x, tol=1e-6, maxiter=100, check_every=1)
    assert it == 1 and err <= atol
    torch.testing.assert_close(x, b, rtol=1e-6, atol=0)


def _batch_offsets(sizes, device):
    return torch.tensor(np.concatenate([[0], np.cumsum(sizes)]), dtype=torch.int32, device=device)


def _spd_np(n, seed, dtype):
    rng = np.random.default_rng(seed)
    q, _ = np.linalg.qr(rng.standard_normal((n, n)))
    A = (q * rng.uniform(1.0, 10.0, n)) @ q.T
    return A.astype(dtype), rng.standard_normal(n).astype(dtype)


@pytest.mark.parametrize("sizes", [[20, 20, 20, 20], [8, 15, 10, 12]])
def test_batched_cg_dense(device, sizes):
    """test_batched_cg / test_batched_nonuniform (test_linear_solvers.py:451-489):
    block-diagonal SPD system, one subproblem per block; each block's residual
    within 32 tol |b_i| (FP32)."""
    rows = sum(sizes)
    A = np.zeros((rows, rows), np.float32)
    b = np.zeros(rows, np.float32)
    off = np.concatenate([[0], np.cumsum(sizes)])
    for i, n in enumerate(sizes):
        A[off[i]:off[i + 1], off[i]:off[i + 1]], b[off[i]:off[i + 1]] = _spd_np(n, i, np.float32)
    op = linear.aslinearoperator(torch.tensor(A, device=device), batch_offsets=_batch_offsets(sizes, device),
                                 max_batch_length=max(sizes))
    assert op.batch_count == len(sizes) and op.max_batch_length == max(sizes)
    x = torch.zeros(rows, device=device)
    it, err, atol = linear.cg(op, torch.tensor(b, device=device), x, tol=1e-5, maxiter=1000)
    assert err <= atol
    xn = x.cpu().numpy().astype(np.float64)
    for i in range(len(sizes)):
        sl = slice(off[i], off[i + 1])
        res = np.linalg.norm(A[sl, sl].astype(np.float64) @ xn[sl] - b[sl])
        assert res <= 32 * 1e-5 * np.linalg.norm(b[sl].astype(np.float64)), i


def test_batched_cg_vector_entries_and_inactive_tail(device):
    """test_batched_vector_offsets / _inactive_tail / _vector_inactive_tail
    (test_linear_solvers.py:492-577): diagonal operators, entries of two scalars
    assigned to the subproblem of their first dof, inactive dofs untouched."""
    d = torch.tensor([2.0, 2.0, 5.0, 5.0], device=device)
    b = torch.tensor([[2.0, 4.0], [10.0, 15.0]], device=device)
    x = torch.zeros_like(b)
    op = linear.aslinearoperator(d, batch_offsets=_batch_offsets([2, 2], device), max_batch_length=2)
    linear.cg(op, b, x, tol=1e-7, maxiter=4, check_every=1, use_cuda_graph=False)
    np.testing.assert_allclose(x.cpu().numpy(), [[1.0, 2.0], [2.0, 3.0]], rtol=1e-5, atol=1e-5)
    # one subproblem over the first three dofs of five
    d = torch.tensor([2.0, 3.0, 4.0, 5.0, 6.0], dtype=torch.float64, device=device)
    b = torch.tensor([2.0, 6.0, 12.0, 100.0, 200.0], dtype=torch.float64, device=device)
    x = torch.tensor([0.0, 0.0, 0.0, 7.0, 8.0], dtype=torch.float64, device=device)
    op = linear.aslinearoperator(d, batch_offsets=_batch_offsets([3], device), max_batch_length=3)
    it, err, atol = linear.cg(op, b, x, tol=1e-8, maxiter=20, check_every=1)
    assert it > 1 and err <= atol
    np.testing.assert_allclose(x.cpu().numpy(), [1.0, 2.0, 3.0, 7.0, 8.0], rtol=1e-7, atol=1e-7)
    # two-scalar entries, the last entry inactive
    d = torch.tensor([2.0, 3.0, 4.0, 5.0, 6.0, 7.0], dtype=torch.float64, device=device)
    b = torch.tensor([[2.0, 6.0], [12.0, 20.0], [100.0, 200.0]], dtype=torch.float64, device=device)
    x = torch.tensor([[0.0, 0.0], [0.0, 0.0], [7.0, 8.0]], dtype=torch.float64, device=device)
    op = linear.aslinearoperator(d, batch_offsets=_batch_offsets([2, 2], device), max_batch_length=2)
    _, err, atol = linear.cg(op, b, x, tol=1e-8, maxiter=8, check_every=1, use_cuda_graph=False)
    assert err <= atol
    np.testing.assert_allclose(x.cpu().numpy(), [[1.0, 2.0], [3.0, 4.0], [7.0, 8.0]], rtol=1e-7, atol=1e-7)


def test_batched_cg_bsr_matches_single_solves(device):
    """Three 2D Poisson systems stacked block-diagonally in one BSR matrix,
    one subproblem each, Jacobi-preconditioned: every subproblem's solution
    equals its own single-system solve (the subproblems only differ in the FP64
    dot grouping) and the device-side results hold one value per subproblem."""
    mats = []
    for k, n in enumerate((12, 16, 20)):
        rows, cols, vals, b, nd = problems.poisson2d_q1(n, k)
        mats.append((rows, cols, vals, b, nd))
    off = np.concatenate([[0], np.cumsum([m[4] for m in mats])])
    R = np.concatenate([m[0] + off[i] * (m[0] >= 0) for i, m in enumerate(mats)]).astype(np.int32)
    C = np.concatenate([m[1] + off[i] * (m[1] >= 0) for i, m in enumerate(mats)]).astype(np.int32)
    R = np.where(np.concatenate([m[0] for m in mats]) < 0, -1, R)
    C = np.where(np.concatenate([m[1] for m in mats]) < 0, -1, C)
    V = np.concatenate([m[2] for m in mats])
    B = np.concatenate([m[3] for m in mats])
    ntot = int(off[-1])
    A = _bsr_from(device, ntot, torch.from_numpy(R), torch.from_numpy(C), torch.from_numpy(V))
    M = linear.preconditioner(A, "diag")
    op = linear.aslinearoperator(A, batch_offsets=torch.tensor(off, dtype=torch.int32, device=device))
    x = torch.zeros(ntot, device=device)
    it, err, atol = linear.cg(op, torch.from_numpy(B).to(device), x, tol=1e-6, maxiter=2000, M=M)
    assert err <= atol
    for i, (rows, cols, vals, b, nd) in enumerate(mats):
        Ai = _bsr_from(device, nd, torch.from_numpy(rows), torch.from_numpy(cols), torch.from_numpy(vals))
        xi = torch.zeros(nd, device=device)
        linear.cg(Ai, torch.from_numpy(b).to(device), xi, tol=1e-6, maxiter=2000, M=linear.preconditioner(Ai, "diag"))
        xs = x[off[i]:off[i + 1]].cpu().numpy()
        ref = xi.cpu().numpy()
        assert np.linalg.norm(xs - ref) <= 1e-4 * np.linalg.norm(ref), i
    x.zero_()
    its, rr, at = linear.cg(op, torch.from_numpy(B).to(device), x, tol=1e-6, maxiter=400, M=M, check_every=0)
    assert rr.shape == (3,) and at.shape == (3,) and bool((rr <= at).all())


@pytest.mark.parametrize("n,restart,check_every", [(64, None, 10), (64, 5, 10), (64, 7, 10), (64, None, 0),
                                                   (600, None, 10)])
def test_cg_graph_replay_matches_eager(device, n, restart, check_every):
    """use_cuda_graph replays the cycles between two checks as one HIP graph
    on a private stream (small systems); the iterates are the eager ones bit
    for bit, replay after replay: fused direction pass with device-side buffer
    parity at n = 64, restart cycles that divide check_every (graphed) or not
    (eager), device-only convergence (groups of 16 cycles), and a large system
    that always launches directly (n = 600).  The callback keeps the small
    systems on the general kernels (without it they are solved in one launch)."""
    rows, cols, vals, b, nd = problems.poisson2d_q1(n, 3)
    A = _bsr_from(device, nd, torch.from_numpy(rows), torch.from_numpy(cols), torch.from_numpy(vals))
    M = linear.preconditioner(A, "diag")
    bt = torch.from_numpy(b).to(device)
    out = []
    for graph in (False, True, True):
        x = torch.zeros_like(bt)
        (it, err, atol), window, finished = _solve_with_route(
            A, bt, x, tol=1e-6, maxiter=3000, M=M, restart=restart, check_every=check_every, use_cuda_graph=graph,
            callback=lambda *a: None)
        assert window == finished == 0
        if check_every == 0:
            it, err = int(it.cpu()[0]), float(err.cpu()[0])
        out.append((it, err, x.cpu().numpy().tobytes()))
    assert out[0] == out[1] == out[2]
    assert out[0][0] > 10


def _seg_dot(device, a, b, offs):
    from warp_amd import _native

    lib = _native.lib()
    n, nb = a.numel(), offs.numel() - 1
    sfx = "f64" if a.dtype == torch.float64 else "f32"
    chunk = torch.empty(nb + 1, dtype=torch.int32, device=device)
    wsb = lib.warp_amd_seg_dot_plan_workspace_size(nb)
    ws = torch.empty(wsb, dtype=torch.uint8, device=device)
    s = torch.cuda.current_stream(device).cuda_stream
    _native.call("warp_amd_seg_dot_plan", nb, offs.data_ptr(), chunk.data_ptr(), ws.data_ptr(), wsb, s)
    mc = lib.warp_amd_seg_dot_max_chunks(n, nb)
    partials = torch.empty(max(mc, 1), dtype=torch.float64, device=device)
    out = torch.full((nb,), float("nan"), dtype=torch.float64, device=device)
    _native.call(f"warp_amd_seg_dot_{sfx}", n, nb, offs.data_ptr(), chunk.data_ptr(), mc, a.data_ptr(), b.data_ptr(),
                 partials.data_ptr(), out.data_ptr(), s)
    return out.cpu().numpy()


def test_segmented_dot_known_answers(device):
    """test_tiled_dot_large_single_batch / _batched_tree known answers
    (test_linear_solvers.py:605-680): inactive tail excluded, empty and odd-sized
    subproblems, and per-subproblem sums against FP64 sums of the same data."""
    length = 100_000
    active = length - 2
    a = torch.full((length,), 2.0, device=device)
    a[active:] = 100.0
    out = _seg_dot(device, a, a, _batch_offsets([active], device))
    assert out[0] == 4 * active
    sizes = [0, 1, 511, 512, 513, 65_537, 262_145]
    n = sum(sizes) + 17
    offs = _batch_offsets(sizes, device)
    two = torch.full((n,), 2.0, device=device)
    three = torch.full((n,), 3.0, device=device)
    np.testing.assert_array_equal(_seg_dot(device, two, three, offs), 6.0 * np.array(sizes))
    rng = np.random.default_rng(123)
    x = rng.standard_normal(n)
    y = rng.standard_normal(n)
    got = _seg_dot(device, torch.tensor(x, device=device), torch.tensor(y, device=device), offs)
    bo = np.concatenate([[0], np.cumsum(sizes)])
    ref = np.array([math.fsum(x[s:e] * y[s:e]) for s, e in zip(bo[:-1], bo[1:])])
    np.testing.assert_allclose(got, ref, rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("prec", ["diag", "id"])
@pytest.mark.parametrize("dtype,n", [(torch.float32, n) for n in (89, 129, 161, 215)] +
                         [(torch.float64, n) for n in (61, 89, 129, 187)])
def test_cg_vector_update_and_wave_spmv(device, dtype, n, prec, shift):
    """Unfused scalar systems: the 16-byte update with its tail (odd n^3), the
    scalar update for an x that is not 16-byte aligned, and each size rule of the
    large systems: lane groups (FP32 89, FP64 61), wave tiles (FP32 from 2^21
    rows: 129; FP64 from 2^19: 89), vectors past the caches (161; 129) and the
    matrix too (more than 512 MB: 215; 187).  Twelve iterations against the same
    recurrence in float64 torch.  Bound: how far rounding grows depends on the
    system (a Ritz value that converges within the twelve iterations makes it
    grow some thousandfold, as an outlier of exp(N(0, 1)) coefficients does without
    a preconditioner; so the other sizes than 89 take exp(N(0, 1/16)), which has
    none), and it is measured on the system: the recurrence once more
    with every sum (of a row, of a vector update, alpha and beta) off by a random
    share of its terms' magnitude, a unit roundoff at most.  The solver rounds each
    of them a few times (seven terms of a row, say), hence within ten times that
    difference; one wrong entry of N gives N^-1/2 > 3e-4."""
    from warp_amd import problems

    g = torch.Generator(device=device).manual_seed(n)
    k = torch.exp((1.0 if n == 89 else 0.25) * torch.randn((n, n, n), generator=g, device=device))
    off, col, val = problems.fv7_poisson(k)
    N = n**3
    A = sparse.bsr_zeros(N, N, wa.types.type_to_scalar(dtype), device=device)
    A.offsets, A.columns, A.values, A.nnz = off, col, val.to(dtype), col.numel()
    b = torch.randn(N, generator=g, device=device, dtype=dtype)
    store = torch.zeros(N + 8, dtype=dtype, device=device)
    x = store[shift:shift + N]
    (it, _, _), window, finished = _solve_with_route(A, b, x, tol=1e-14, atol=0.0, maxiter=12,
                                                     M=linear.preconditioner(A, prec))
    assert window == finished == 0  # not one launch
    assert it == 12 and float(store[N + shift:].abs().max()) == 0.0
    rows = torch.repeat_interleave(torch.arange(N, device=device), (off[1:] - off[:-1]).long())
    v64, c64 = val.double(), col.long()

    def mv(v, u):
        return torch.zeros(N, dtype=torch.float64, device=device).index_add(0, rows, v * u[c64])

    inv = 1.0 / v64[rows == c64] if prec == "diag" else torch.ones(N, dtype=torch.float64, device=device)

    def recurrence(u, seed):
        """x after twelve iterations, every sum off by a random share u of its terms' magnitude at most."""
        noise = torch.Generator(device=device).manual_seed(seed)

        def add(*terms):
            t = sum(terms)
            if u == 0.0:
                return t
            off = 2.0 * torch.rand(t.shape, generator=noise, device=device, dtype=torch.float64) - 1.0
            return t + u * off * sum(v.abs() for v in terms)

        xs = torch.zeros(N, dtype=torch.float64, device=device)
        r = b.double()
        z = add(inv * r)
        p, rz = z, r @ z
        for _ in range(12):
            q = mv(v64, p)
            if u:
                q = q + (add(torch.ones_like(q)) - 1.0) * mv(v64.abs(), p.abs())
            a = add(rz / (p @ q))
            xs, r = add(xs, a * p), add(r, -a * q)
            z = add(inv * r)
            rz, old = r @ z, rz
            p = add(z, add(rz / old) * p)
        return xs

    u = 2.0**-24 if dtype == torch.float32 else 2.0**-53
    xs = recurrence(0.0, 0)
    rel = float((x.double() - xs).norm() / xs.norm())
    grown = max(float((recurrence(u, seed) - xs).norm() / xs.norm()) for seed in (1, 2))
    print(f"[cg large] {n}^3 {dtype} {prec}: relative difference {rel:.2e}, of perturbed recurrences {grown:.2e}")
    assert rel < 10.0 * max(grown, u) < 3e-4, (rel, grown)


@pytest.mark.parametrize("prec", ["diag", "block_diag", "id"])
@pytest.mark.parametrize("family,n,dtype", [
    ("poisson", 3, torch.float32), ("poisson", 24, torch.float32), ("poisson", 200, torch.float32),
    ("poisson", 90, torch.float64), ("elasticity", 3, torch.float32), ("elasticity", 9, torch.float64),
    ("elasticity", 17, torch.float32), ("renumbered", 200, torch.float32)])
def test_cg_one_launch_solve(device, family, n, dtype, prec):
    """Small systems in one launch (one workgroup up to the most, rows that do
    not divide, windows that do not fit: a random numbering) against the same
    solve with a callback, which takes the general kernels: same iteration count
    (whole groups of check_every, maxiter).  Only the order of the FP64 sums
    differs.  Over 12 iterations the iterates agree to 1e-5 (FP32 rounds alpha and
    beta once per iteration: 12 * 6e-8, grown by less than 10) and 1e-12 (FP64:
    12 * 1e-16 and the same growth leave 1e-14); later ones part as Ritz values
    converge, so a converged solve is held to the other's true residual."""
    if family == "elasticity":
        r, c, v, b, nn = problems.elasticity3d_q1(n, device=device)
        A = sparse.bsr_zeros(nn, nn, wa.matrix((3, 3), wa.types.type_to_scalar(dtype)), device=device)
        sparse.bsr_set_from_triplets(A, r, c, v.to(dtype), prune_numerical_zeros=False)
    else:
        r, c, v, b, nn = problems.poisson2d_q1(n, 1)
        r, c, v, b = (torch.from_numpy(t).to(device) for t in (r, c, v, b))
        if family == "renumbered":
            perm = torch.randperm(nn, generator=torch.Generator().manual_seed(1)).to(device)
            keep = (r >= 0) & (c >= 0)
            r, c, v = perm[r[keep].long()].to(torch.int32), perm[c[keep].long()].to(torch.int32), v[keep]
            b = torch.empty_like(b).index_copy_(0, perm, b)
        A = sparse.bsr_zeros(nn, nn, wa.types.type_to_scalar(dtype), device=device)
        sparse.bsr_set_from_triplets(A, r, c, v.to(dtype))
    A.nnz_sync()
    b = b.to(dtype)
    M = linear.preconditioner(A, prec)
    for kw in (dict(tol=1e-12, maxiter=12), dict(tol=1e-5, maxiter=600), dict(tol=1e-5, maxiter=600, check_every=7),
               dict(tol=1e-12, maxiter=37), dict(tol=2.0, maxiter=50)):
        x0, x1 = torch.full_like(b, 0.01), torch.full_like(b, 0.01)
        seen = []
        i0, _, a0 = linear.cg(A, b, x0, atol=0.0, M=M, callback=lambda *a: seen.append(a), **kw)
        i1, e1, a1 = linear.cg(A, b, x1, atol=0.0, M=M, **kw)
        assert i0 == i1 and a0 == a1 and len(seen) > 0
        if kw["maxiter"] == 12:
            tight = 1e-12 if dtype == torch.float64 else 1e-5
            assert float((x0 - x1).norm()) <= tight * float(x0.norm())
        elif e1 <= a1:
            true = [float((b.double() - sparse.bsr_mv(A, x).double()).norm()) for x in (x0, x1)]
            assert true[1] <= 2.0 * true[0] + a1  # the same attainable accuracy


def test_cg_one_launch_nan_and_concurrent_streams(device):
    """A right-hand side with a NaN runs to maxiter as the general kernels do, and
    solves on several streams and threads at once give the serial result."""
    import threading

    r, c, v, b, nn = problems.poisson2d_q1(96, 1)
    A = sparse.bsr_zeros(nn, nn, wa.float32, device=device)
    sparse.bsr_set_from_triplets(A, *(torch.from_numpy(t).to(device) for t in (r, c, v)))
    A.nnz_sync()
    M = linear.preconditioner(A, "diag")
    bt = torch.from_numpy(b).to(device)
    bad = bt.clone()
    bad[5] = float("nan")
    it, err, _ = linear.cg(A, bad, torch.zeros_like(bt), tol=1e-5, maxiter=30, M=M)
    assert it == 30 and math.isnan(err)
    want = torch.zeros_like(bt)
    i0, _, _ = linear.cg(A, bt, want, tol=1e-6, maxiter=200, M=M)
    torch.cuda.synchronize()
    results = [None] * 4

    def work(k):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(5):
                x = torch.zeros_like(bt)
                i, _, _ = linear.cg(A, bt, x, tol=1e-6, maxiter=200, M=M)
            s.synchronize()
        results[k] = (i, x)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i, x in results:
        assert i == i0 and torch.equal(x, want)


def _renumbered_poisson(n, device):
    r, c, v, b, nn = problems.poisson2d_q1(n, 1)
    r, c, v, b = (torch.from_numpy(t).to(device) for t in (r, c, v, b))
    perm = torch.randperm(nn, generator=torch.Generator().manual_seed(1)).to(device)
    keep = (r >= 0) & (c >= 0)
    A = sparse.bsr_zeros(nn, nn, wa.float32, device=device)
    sparse.bsr_set_from_triplets(A, perm[r[keep].long()].to(torch.int32), perm[c[keep].long()].to(torch.int32), v[keep])
    A.nnz_sync()
    return A, torch.empty_like(b).index_copy_(0, perm, b)


@pytest.mark.parametrize("n", [128, 200])
def test_cg_window_misfit_starts_once(device, n):
    """A small system whose columns' window is too large for one launch (a random
    numbering; at 128 it fits the LDS, but is slower so) goes on from the state and residual it has (the plan's window is
    still in the state, which initialising again would clear), with the bits of
    the general kernels."""
    A, b = _renumbered_poisson(n, device)
    M = linear.preconditioner(A, "diag")
    runs = []
    for kw in (dict(), dict(callback=lambda *a: None)):
        x = torch.full_like(b, 0.01)
        res, window, finished = _solve_with_route(A, b, x, tol=1e-5, atol=0.0, maxiter=60, M=M, **kw)
        runs.append((res, x.cpu().numpy().tobytes()))
        assert finished == 0
        assert (window > 0) == (not kw)
    assert runs[0] == runs[1]


def _on_streams(jobs):
    """Each job on a thread and stream of its own; their results."""
    import threading

    out = [None] * len(jobs)

    def work(k):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            out[k] = jobs[k]()
        s.synchronize()

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    return out


def test_cg_one_launch_solves_overlap(device):
    """One-launch solves of several sizes on eight streams at once, more
    workgroups than may be in flight together: each has the bits of its serial
    solve and none fell back.  And they overlap: four streams take less than 2.6
    times as long as one for four times the solves (measured 1.7; 3.4 when the
    launches ran one after another)."""
    import time

    def system(n, dtype):
        r, c, v, b, nn = problems.poisson2d_q1(n, 1)
        A = sparse.bsr_zeros(nn, nn, wa.types.type_to_scalar(dtype), device=device)
        sparse.bsr_set_from_triplets(A, torch.from_numpy(r).to(device), torch.from_numpy(c).to(device),
                                     torch.from_numpy(v).to(device, dtype))
        A.nnz_sync()
        return A, torch.from_numpy(b).to(device, dtype), linear.preconditioner(A, "diag")

    def solve(A, b, M, repeat):
        for _ in range(repeat):
            x = torch.zeros_like(b)
            res, _, finished = _solve_with_route(A, b, x, tol=1e-30, atol=0.0, maxiter=80, M=M)
        return res, finished, x

    systems = [system(n, dt) for n in (250, 17, 128, 200) for dt in (torch.float32, torch.float64)]
    serial = [solve(*s, 1) for s in systems]
    torch.cuda.synchronize()
    together = _on_streams([lambda s=s: solve(*s, 6) for s in systems])
    for (r0, f0, x0), (r1, f1, x1) in zip(serial, together):
        assert r0 == r1 and f0 == f1 and f1 > 0 and torch.equal(x0, x1)
    A, b, M = systems[4]

    def many():
        mine = linear.cg(A, b, torch.zeros_like(b), tol=1e-30, atol=0.0, maxiter=80, M=M, run=False)
        for _ in range(40):
            mine()

    took = {}
    for threads in (1, 4) * 4:
        torch.cuda.synchronize()
        t = time.perf_counter()
        _on_streams([many] * threads)
        took[threads] = min(took.get(threads, math.inf), time.perf_counter() - t)
    print(f"[cg one-launch] 40 solves each: 1 stream {took[1] * 1e3:.1f} ms, 4 streams {took[4] * 1e3:.1f} ms")
    assert took[4] < 2.6 * took[1]


@pytest.mark.parametrize("polls,maxiter", [(0, 1), (0, 60), (1, 1), (1, 60), (3, 60)])
@pytest.mark.parametrize("family,n,dtype", [("poisson", 90, torch.float32), ("elasticity", 9, torch.float64)])
def test_cg_one_launch_falls_back(device, family, n, dtype, polls, maxiter):
    """A one-launch solve whose waits run out (a limit of a few looks at the
    others' sums: every workgroup leaves by itself, some after iterations of
    their own) leaves x alone, and the general kernels give the bits they give
    with a callback; if all looks succeeded, the one-launch solve's."""
    import ctypes

    from warp_amd import _native

    if family == "elasticity":
        r, c, v, b, nn = problems.elasticity3d_q1(n, device=device)
        btype = wa.matrix((3, 3), wa.types.type_to_scalar(dtype))
    else:
        r, c, v, b, nn = problems.poisson2d_q1(n, 1)
        r, c, v, b = (torch.from_numpy(t).to(device) for t in (r, c, v, b))
        btype = wa.types.type_to_scalar(dtype)
    A = sparse.bsr_zeros(nn, nn, btype, device=device)
    sparse.bsr_set_from_triplets(A, r, c, v.to(dtype))
    A.nnz_sync()
    b = b.to(dtype)
    M = linear.preconditioner(A, "diag")
    want = []
    for kw in (dict(), dict(callback=lambda *a: None)):
        x = torch.full_like(b, 0.01)
        res, _, finished = _solve_with_route(A, b, x, tol=1e-30, atol=0.0, maxiter=maxiter, M=M, **kw)
        want.append((finished, res, x))
    assert want[0][0] > 1 and want[1][0] == 0
    lib = _native.lib()
    x = torch.full_like(b, 0.01)
    ws = torch.empty(lib.warp_amd_cg_workspace_size(x.numel(), x.element_size()), dtype=torch.uint8, device=device)
    it, err, atol = ctypes.c_int(0), ctypes.c_double(0.0), ctypes.c_double(0.0)
    _native.call("warp_amd_cg_solve_polls_f64" if dtype == torch.float64 else "warp_amd_cg_solve_polls_f32", nn,
                 A.block_shape[0], A.offsets.data_ptr(), A.columns.data_ptr(), A.values.data_ptr(), int(A.nnz),
                 linear.PREC_DIAG, M._prec_data.data_ptr(), b.data_ptr(), x.data_ptr(), 1e-30, 0.0, maxiter, 10, polls,
                 ws.data_ptr(), ws.numel(), ctypes.byref(it), ctypes.byref(err), ctypes.byref(atol),
                 _native.stream_of(device))
    o = lib.warp_amd_cg_state_offset(4)
    finished = int(ws[o:o + 4].view(torch.int32))
    print(f"[cg fallback] {family} polls {polls}: {finished} workgroups finished after the solve's last start")
    assert finished in (0, want[0][0]) and (polls > 0 or finished == 0)
    _, res, xw = want[0] if finished else want[1]
    assert (it.value, err.value, atol.value) == res and torch.equal(x, xw)
