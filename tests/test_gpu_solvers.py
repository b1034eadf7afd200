"""Reductions, BLAS-1 and the Krylov solvers on the GPU through the C ABI, against the oracle
(single-thread TNL semantics, pinned to TNL's own residual histories) and the mathematics."""
import os
import time
import numpy as np
import pytest
import torch

import pyoracle as O
import workloads as W

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.gpu


def t(a, dev, dt=torch.float64):
    return torch.tensor(np.asarray(a), dtype=dt, device=dev)


def test_dot_norm_closed_forms_and_determinism(tnl, dev):
    # reduceTest.h:91-128 closed forms; same bits on repeated calls
    for size in [1, 2, 127, 128, 255, 256, 257, 1000, 9377, 100000, 4096000]:
        ones = torch.ones(size, dtype=torch.float64, device=dev)
        assert tnl.dot(ones, ones) == size
        iota = torch.arange(size, dtype=torch.float64, device=dev)
        assert tnl.dot(iota, ones) == size * (size - 1) / 2
    rng = np.random.default_rng(1)
    a = rng.standard_normal(1 << 20)
    b = rng.standard_normal(1 << 20)
    ad, bd = t(a, dev), t(b, dev)
    d1 = tnl.dot(ad, bd)
    assert all(tnl.dot(ad, bd) == d1 for _ in range(5))
    assert abs(d1 - float(np.dot(a, b))) <= 1e-12 * float(np.abs(a) @ np.abs(b))
    assert abs(tnl.lpNorm2(ad) - np.linalg.norm(a)) <= 1e-13 * np.linalg.norm(a)
    a32 = t(a, dev, torch.float32)
    assert abs(tnl.dot(a32, a32) - float(np.dot(a.astype(np.float32).astype(np.float64),
                                                 a.astype(np.float32).astype(np.float64)))) < 1e-9 * len(a)


def test_axpby_multidot_gemv_scan(tnl, dev):
    rng = np.random.default_rng(2)
    n, k = 100003, 31
    ld = ((n + 31) // 32) * 32
    V = rng.standard_normal((k, ld))
    w = rng.standard_normal(n)
    Vd, wd = t(V.ravel(), dev), t(w, dev)
    got = tnl.multidot(Vd, ld, k, wd)
    want = V[:, :n] @ w
    assert np.all(np.abs(got - want) <= 1e-12 * (np.abs(V[:, :n]) @ np.abs(w)))
    c = rng.standard_normal(20)
    y = rng.standard_normal(n)
    yd = t(y, dev)
    tnl.gemv(-1.0, Vd, ld, 20, c, 0.5, yd)
    want = -(V[:20, :n].T @ c) + 0.5 * y
    np.testing.assert_allclose(yd.cpu().numpy(), want, rtol=1e-12, atol=1e-12)
    x = rng.standard_normal(n)
    yd = t(y, dev)
    tnl.axpby(2.0, t(x, dev), -3.0, yd)
    np.testing.assert_allclose(yd.cpu().numpy(), 2 * x - 3 * y, rtol=1e-15, atol=1e-15)
    caps = rng.integers(0, 50, 1234567).astype(np.int32)
    cd = torch.tensor(caps, device=dev)
    out = torch.zeros(len(caps) + 1, dtype=torch.int32, device=dev)
    tnl.exclusive_scan(cd, out)
    want = np.zeros(len(caps) + 1, np.int64)
    np.cumsum(caps, out=want[1:])
    np.testing.assert_array_equal(out.cpu().numpy(), want.astype(np.int32))


def _run_device_solver(tnl, dev, method, rp, c, v, b, fmt="CSRLight", dtype="f64", **params):
    A = tnl.SparseMatrix.from_csr(rp, c, v, format=fmt, dtype=dtype)
    s = tnl.getLinearSolver(method)
    s.setMatrix(A)
    s.setup(**params)
    bd = t(b, dev, A.vector_dtype)
    xd = torch.zeros(len(b), dtype=A.vector_dtype, device=dev)
    ok = s.solve(bd, xd)
    return ok, s.getIterations(), s.getResidue(), s.getResidualHistory(), xd.cpu().numpy().astype(np.float64)


def test_solvers_follow_tnl_histories(tnl, golden, dev):
    """Every fixture run (CG, BiCGStab, all GMRES variants, with and without Jacobi): same
    convergence flag, iteration count within 2 of the range TNL's own count spans over OpenMP
    thread counts, residual history within 1e-6 relative over the first iterations (the device
    sums in a different order), true residual at the tolerance."""
    d = golden["solvers"]
    runs = sorted({k.split("/")[0] for k in d.files if k.startswith("run")})
    errors = []
    for run in runs:
        try:
            _check_run(tnl, d, dev, run)
        except AssertionError as e:
            errors.append(f"{run}: {e}")
    assert not errors, "\n".join(errors)


def _check_run(tnl, d, dev, run):
    sysname = str(d[f"{run}/system"])
    method = str(d[f"{run}/method"])
    params = dict(eval(str(d[f"{run}/params"])))
    print(f"run {run} {sysname} {method} {params}", flush=True)
    rp, c, v, b = (d[f"{sysname}/{k}"] for k in ("row_ptr", "cols", "vals", "b"))
    ok, its, res, hist, x = _run_device_solver(tnl, dev, method, rp, c, v, b, **params)
    ref_its = int(d[f"{run}/iterations"][0])
    assert ok == bool(d[f"{run}/converged"][0]), run
    # within 2 (ell for BiCGStab(ell)) of TNL's count, or of the range TNL's own count spans over
    # OpenMP thread counts: BiCGStab on the 2D Laplacian moves by up to 10 iterations with the
    # reduction order of its dot products alone
    spread = d[f"{run}/iterations_threads"]
    slack = max(2, params.get("bicgstab_ell", 1))
    assert min(spread) - slack <= its <= max(spread) + slack, (run, its, ref_its, list(spread))
    h_ref = d[f"{run}/history"]
    m = min(len(hist), len(h_ref), 20)
    # residues near 1e-12 and below are exact residues b - A x at the rounding floor of A x
    # (about 1e-16 |A| |x| / |b|), hence the absolute 1e-14
    np.testing.assert_allclose(hist[:m], h_ref[:m], rtol=1e-6, atol=1e-14, err_msg=run)
    A = W.csr_to_dense(rp, c, v, len(b))
    true_res = np.linalg.norm(b - A @ x) / np.linalg.norm(b)
    tol = params.get("convergence_residue", 1e-6)
    assert true_res < 50 * tol, (run, true_res)


def test_cg_laplacian_2d_256_config(tnl, dev):
    """The CPU configuration: 256^2 5-point Laplacian, CG to 1e-8 from x0 = 0 (756 iterations on
    TNL's Host path for its seed); device and oracle agree on the iteration count."""
    rp, c, v = W.laplacian_2d(256)
    b = W.uniform_vector(len(rp) - 1, 42)
    ref = O.solve("cg", rp, c, v, b, convergence_residue=1e-8, max_iterations=5000)
    ok, its, res, hist, x = _run_device_solver(tnl, dev, "cg", rp, c, v, b, convergence_residue=1e-8,
                                               max_iterations=5000)
    assert ok and abs(its - ref["iterations"]) <= 3
    assert res < 1e-8
    np.testing.assert_allclose(hist[:50], ref["history"][:50], rtol=1e-8)


@pytest.mark.parametrize("fmt", ["CSRScalar", "CSRAdaptive", "Ellpack", "SlicedEllpack", "ChunkedEllpack", "BiEllpack"])
def test_solvers_independent_of_format(tnl, dev, fmt):
    rp, c, v = W.convection_diffusion_3d(10, 10.0)
    b = W.uniform_vector(len(rp) - 1, 3)
    ok, its, res, hist, x = _run_device_solver(tnl, dev, "bicgstab", rp, c, v, b, fmt=fmt, convergence_residue=1e-10,
                                               max_iterations=2000, preconditioner=1)
    ref = O.solve("bicgstab", rp, c, v, b, convergence_residue=1e-10, max_iterations=2000, preconditioner=1)
    assert ok and abs(its - ref["iterations"]) <= 2


def test_failure_paths(tnl, dev):
    """max_iterations reached -> solve() is false; NaN in b -> false; b = 0 -> immediate
    convergence with x = 0 (normb := 1, CG.hpp:32-33)."""
    rp, c, v = W.laplacian_2d(32)
    n = len(rp) - 1
    b = W.uniform_vector(n, 1)
    ok, its, *_ = _run_device_solver(tnl, dev, "cg", rp, c, v, b, convergence_residue=1e-12, max_iterations=5)
    assert not ok
    ref = O.solve("cg", rp, c, v, b, convergence_residue=1e-12, max_iterations=5)
    assert its == ref["iterations"]
    bn = b.copy()
    bn[7] = np.nan
    ok, *_ = _run_device_solver(tnl, dev, "gmres", rp, c, v, bn, convergence_residue=1e-8, max_iterations=100)
    assert not ok
    ok, its, res, hist, x = _run_device_solver(tnl, dev, "bicgstab", rp, c, v, np.zeros(n), convergence_residue=1e-8)
    assert ok and np.all(x == 0)


def test_float32_solve(tnl, dev):
    rp, c, v = W.laplacian_3d(16)
    b = W.uniform_vector(len(rp) - 1, 9)
    ok, its, res, hist, x = _run_device_solver(tnl, dev, "cg", rp, c, v, b, dtype="f32", convergence_residue=1e-5,
                                               max_iterations=1000)
    ref = O.solve("cg", rp, c, v, b, convergence_residue=1e-5, max_iterations=1000)
    assert ok and abs(its - ref["iterations"]) <= 3


@pytest.mark.parametrize("method,precond", [("cg", 0), ("cg", 1), ("bicgstab", 1), ("tfqmr", 0), ("tfqmr", 1),
                                            ("cg", 2), ("bicgstab", 2), ("bicgstabl", 1)])
def test_graph_replay_matches_direct_launches(tnl, dev, method, precond):
    """Iterations replayed from a captured hipGraph give the same bits as the same kernels
    launched one by one (long enough to go past the eager batches)."""
    rp, c, v = W.laplacian_3d(24) if method in ("cg", "tfqmr") else W.convection_diffusion_3d(20, 10.0)
    b = W.uniform_vector(len(rp) - 1, 4)
    runs = []
    for g in (0, 1):
        ok, its, res, hist, x = _run_device_solver(tnl, dev, method, rp, c, v, b, convergence_residue=1e-10,
                                                   max_iterations=3000, preconditioner=precond, use_graph=g)
        runs.append((ok, its, res, hist, x))
    assert runs[0][1] > 16  # past the eager chunks of 4 and 8 iterations
    assert runs[0][0] == runs[1][0] and runs[0][1] == runs[1][1]
    np.testing.assert_array_equal(runs[0][4], runs[1][4])
    np.testing.assert_array_equal(runs[0][3], runs[1][3])


def _restart_blocks(m):
    """m copies of a 3x3 system whose residual after one BiCGStab step is exactly orthogonal to r*,
    so that the restart (BICGStab.hpp:88-95) is taken at once."""
    block = np.array([[2.0, 1.0, -1.0], [1.0, 3.0, 1.0], [1.0, -1.0, 2.0]])
    rp = np.arange(3 * m + 1, dtype=np.int32) * 3
    cols = (np.repeat(np.arange(m), 9) * 3 + np.tile(np.tile([0, 1, 2], 3), m)).astype(np.int32)
    return rp, cols, np.tile(block.ravel(), m), np.tile([1.0, 0.0, 0.0], m)


@pytest.mark.parametrize("fmt", ["CSRScalar", "CSRAdaptive", "Ellpack", "SlicedEllpack", "ChunkedEllpack", "BiEllpack"])
@pytest.mark.parametrize("n", [1, 2, 63, 257, 1025, 4097, 70001])
def test_fused_iterations_follow_the_oracle(tnl, dev, fmt, n):
    # tridiagonal, nonsymmetric for BiCGStab: sizes around wavefronts, workgroups, 16-byte lanes and
    # partial counts; x at an odd 8-byte offset, so that the passes' narrow loads run
    for method in ("cg", "bicgstab"):
        up = -1.0 if method == "cg" else -0.7
        i = np.arange(n)
        r = np.concatenate([i[1:], i, i[:-1]])
        c = np.concatenate([i[1:] - 1, i, i[:-1] + 1])
        v = np.concatenate([np.full(n - 1, -1.0), 2.2 + 0.3 * np.cos(i), np.full(n - 1, up)])
        o = np.lexsort((c, r))
        rp = np.zeros(n + 1, np.int32)
        np.cumsum(np.bincount(r, minlength=n), out=rp[1:])
        cols, vals = c[o].astype(np.int32), v[o]
        b = W.uniform_vector(n, 11)
        for pre in (0, 1):
            p = dict(convergence_residue=1e-10, max_iterations=60, preconditioner=pre)
            ref = O.solve(method, rp, cols, vals, b, **p)
            A = tnl.SparseMatrix.from_csr(rp, cols, vals, format=fmt, dtype="f64")
            s = tnl.getLinearSolver(method)
            s.setMatrix(A)
            s.setup(**p)
            bd, xd = t(b, dev), torch.zeros(n + 1, dtype=torch.float64, device=dev)[1:]
            s.solve(bd, xd)
            h = s.getResidualHistory()
            # up to where the residual is rounding alone (one or two rows are solved in as many steps,
            # and what is left may be 0, so the oracle's BiCGStab divides 0 by 0)
            with np.errstate(invalid="ignore"):
                m = min(12, int(np.argmin(np.append(ref["history"] > 1e-13, False))))
            assert len(h) >= m >= 1
            # the sums of up to 70001 products in another order: 1e-13 each, amplified by the steps
            np.testing.assert_allclose(h[:m], ref["history"][:m], rtol=1e-8, atol=1e-14)
            if n <= 2:
                continue
            assert abs(s.getIterations() - ref["iterations"]) <= 1
            np.testing.assert_allclose(xd.cpu().numpy(), ref["x"], rtol=0, atol=1e-8 * np.abs(ref["x"]).max())


def _follow(tnl, dev, rp, cols, vals, fmt, dt, steps, method, pre, rtol):
    """The first residuals of a solve follow the oracle's; x at an odd element offset."""
    b = W.uniform_vector(len(rp) - 1, 11)
    p = dict(convergence_residue=1e-30, max_iterations=steps, preconditioner=pre)
    ref = O.solve(method, rp, cols, vals, b, **p)
    A = tnl.SparseMatrix.from_csr(rp, cols, vals, format=fmt, dtype=dt)
    s = tnl.getLinearSolver(method)
    s.setMatrix(A)
    s.setup(**p)
    x = torch.zeros(len(b) + 1, dtype=A.vector_dtype, device=dev)[1:]
    s.solve(t(b, dev, A.vector_dtype), x)
    h = s.getResidualHistory()
    assert len(h) >= steps and s.getIterations() == ref["iterations"]
    np.testing.assert_allclose(h[:steps], ref["history"][:steps], rtol=rtol)
    np.testing.assert_allclose(x.cpu().numpy(), ref["x"], rtol=0, atol=rtol * np.abs(ref["x"]).max())


@pytest.mark.parametrize("method", ["cg", "bicgstab"])
@pytest.mark.parametrize("fmt,dt,n", [("CSRScalar", "f64", 299999), ("CSRScalar", "f64", 600001), ("CSRScalar", "f32", 299999),
                                      ("SlicedEllpack", "f64", 600001), ("SlicedEllpack", "f32", 70001),
                                      ("SlicedEllpack", "f32", 600001), ("Ellpack", "f32", 300001),
                                      ("ChunkedEllpack", "f32", 70001)])
def test_large_and_single_precision_fused_solves_follow_the_oracle(tnl, dev, method, fmt, dt, n):
    # 299999 CSR rows: 1172 partials, more than a fold loads ahead, with the operand formed in the product; beyond 300000
    # rows the direction has a pass of its own; FP32: four-wide lanes with one, two or three entries left over
    i = np.arange(n)
    r, c = np.concatenate([i[1:], i, i[:-1]]), np.concatenate([i[1:] - 1, i, i[:-1] + 1])
    up = -1.0 if method == "cg" else -0.7
    v = np.concatenate([np.full(n - 1, -1.0), 2.6 + 0.3 * np.cos(i), np.full(n - 1, up)])
    o = np.lexsort((c, r))
    rp = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(r, minlength=n), out=rp[1:])
    for pre in (0, 1):
        # FP64: sums of 600001 products in another order, 1e-13 each, amplified by the steps; FP32: six steps that round
        # vectors of a system of condition 5 at 6e-8
        _follow(tnl, dev, rp, c[o].astype(np.int32), v[o], fmt, dt, 10 if dt == "f64" else 6, method, pre,
                1e-8 if dt == "f64" else 1e-4)


@pytest.mark.parametrize("method", ["cg", "bicgstab"])
@pytest.mark.parametrize("fmt", ["CSRAdaptive", "CSRVector", "CSRLight", "Ellpack", "SlicedEllpack", "ChunkedEllpack", "BiEllpack"])
@pytest.mark.parametrize("dt", ["f64", "f32"])
def test_fused_solves_of_long_rows_follow_the_oracle(tnl, dev, method, fmt, dt):
    # 30 entries a row on average, some rows of 700 (a wavefront's in CSRAdaptive) and of 2600 (a workgroup's)
    n = 4099
    rng = np.random.default_rng(7)
    L = np.full(n, 14)
    L[[5, 900, 4000]] = 700
    L[[77, 78, 2500]] = 2600
    r = np.repeat(np.arange(n), L)
    c = np.concatenate([rng.choice(n, k, replace=False) for k in L])
    w = rng.uniform(-1, 1, len(r))
    key, first = np.unique(np.concatenate([r * n + c, c * n + r]), return_index=True)
    v = np.concatenate([w, w])[first]
    r, c = key // n, key % n
    v[r == c] = 0.0
    v[(r == c)] = 1.0 + np.bincount(r, weights=np.abs(v), minlength=n)[r[r == c]]
    if method == "cg":  # one value for both halves
        v = np.where(r > c, 0.0, v)
        low = np.searchsorted(key, c * n + r)
        v = np.where(r > c, v[low], v)
        v[r == c] = 1.0 + np.bincount(r[r != c], weights=np.abs(v[r != c]), minlength=n)[r[r == c]]
    missing = np.setdiff1d(np.arange(n), r[r == c])  # rows without a diagonal entry get one
    extra = 1.0 + np.bincount(r[r != c], weights=np.abs(v[r != c]), minlength=n)[missing]
    r, c, v = np.concatenate([r, missing]), np.concatenate([c, missing]), np.concatenate([v, extra])
    o = np.lexsort((c, r))
    rp = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(r, minlength=n), out=rp[1:])
    for pre in (0, 1):
        # FP32: rows of 34 products on average round at 34 * 6e-8 of the residual before, up to 20 times the new one, four
        # times over
        _follow(tnl, dev, rp, c[o].astype(np.int32), v[o], fmt, dt, 6 if dt == "f64" else 4, method, pre,
                1e-8 if dt == "f64" else 5e-4)


@pytest.mark.parametrize("method,n", [("cg", 100000), ("cg", 100001), ("bicgstab", 100001)])
def test_rows_of_64_lanes_on_both_sides_of_the_fused_limit(tnl, dev, method, n):
    i = np.arange(n)
    d = [k for k in range(-6, 7)]
    r = np.concatenate([i[max(0, -k):n - max(0, k)] for k in d])
    c = np.concatenate([i[max(0, -k):n - max(0, k)] + k for k in d])
    v = np.where(r == c, 14.0, -1.0 / (1 + np.abs(r - c)))
    if method == "bicgstab":
        v = np.where(c > r, 0.7 * v, v)
    o = np.lexsort((c, r))
    rp = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(r, minlength=n), out=rp[1:])
    # (four steps: the residual falls 150 times a step)
    _follow(tnl, dev, rp, c[o].astype(np.int32), v[o], "CSRVector", "f64", 4, method, 1, 1e-8)


def _arrow(n, m):
    """Tridiagonal with m more entries in row 0 and column 0, symmetric and diagonally dominant."""
    i = np.arange(n)
    e = np.sort(np.random.default_rng(1).choice(np.arange(2, n), m, replace=False))
    r = np.concatenate([i[1:], i, i[:-1], np.zeros(m, int), e])
    c = np.concatenate([i[1:] - 1, i, i[:-1] + 1, e, np.zeros(m, int)])
    d = np.full(n, 4.0)
    d[0] += 1e-3 * m
    v = np.concatenate([np.full(n - 1, -1.0), d, np.full(n - 1, -1.0), np.full(2 * m, 1e-3)])
    o = np.lexsort((c, r))
    rp = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(r, minlength=n), out=rp[1:])
    return rp, c[o].astype(np.int32), v[o]


@pytest.mark.parametrize("method,products", [("cg", 1), ("bicgstab", 2)])
def test_one_long_row_among_short_ones_keeps_its_kernel(tnl, dev, method, products):
    """A solve over CSRAdaptive splits a long row over a workgroup as its product does: an iteration costs about
    two products each (its vector passes included); walked by one lane the row alone costs about 60."""
    rp, c, v = _arrow(200000, 20000)
    n = len(rp) - 1
    A = tnl.SparseMatrix.from_csr(rp, c, v, format="CSRAdaptive", dtype="f64")
    b = t(W.uniform_vector(n, 2), dev)
    y = torch.zeros_like(b)
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    A.vectorProduct(b, y)
    e0.record()
    for _ in range(10):
        A.vectorProduct(b, y)
    e1.record()
    e1.synchronize()
    product = e0.elapsed_time(e1) / 10
    s = tnl.getLinearSolver(method)
    s.setMatrix(A)
    s.setup(convergence_residue=1e-300, max_iterations=8)
    best = 1e9
    for _ in range(3):
        x = torch.zeros_like(b)
        torch.cuda.synchronize()
        start = time.perf_counter()
        s.solve(b, x)
        best = min(best, 1e3 * (time.perf_counter() - start))
    assert best / s.getIterations() < 12 * products * product, (best, product)
    ref = O.solve(method, rp, c, v, b.cpu().numpy(), convergence_residue=1e-300, max_iterations=8)
    # sums of 200000 and of 20000 products in another order: 1e-13 each, amplified by the steps
    np.testing.assert_allclose(s.getResidualHistory()[:6], ref["history"][:6], rtol=1e-8)


@pytest.mark.parametrize("m", [1, 700, 110000])  # the last beyond the rows whose operand the product forms
@pytest.mark.parametrize("use_graph", [0, 1])
def test_bicgstab_restart_follows_the_oracle(tnl, dev, m, use_graph):
    rp, cols, vals, b = _restart_blocks(m)
    p = dict(convergence_residue=1e-12, max_iterations=40)
    ref = O.solve("bicgstab", rp, cols, vals, b, **p)
    ok, its, _, h, x = _run_device_solver(tnl, dev, "bicgstab", rp, cols, vals, b, fmt="SlicedEllpack",
                                          use_graph=use_graph, **p)
    k = min(len(h), len(ref["history"]), 4)  # the steps before the residual is at rounding level
    np.testing.assert_allclose(h[:k], ref["history"][:k], rtol=1e-9, atol=1e-13)
    assert abs(its - ref["iterations"]) <= 1 and ok == bool(ref["converged"])


@pytest.mark.parametrize("restart", [1, 2, 6, 7, 8, 14, 15, 16, 30, 31])
@pytest.mark.parametrize("n", [40, 257, 4913])
def test_cwy_steps_follow_the_oracle(tnl, dev, restart, n):
    # restart lengths around the column buckets of the step's sums (8, 16, 32); sizes about a workgroup
    i = np.arange(n)
    r = np.concatenate([i[1:], i, i[:-1]])
    c = np.concatenate([i[1:] - 1, i, i[:-1] + 1])
    v = np.concatenate([np.full(n - 1, -1.3), 2.5 + 0.2 * np.cos(i), np.full(n - 1, -0.8)])
    o = np.lexsort((c, r))
    rp = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(r, minlength=n), out=rp[1:])
    b = W.uniform_vector(n, 3)
    for pre in (0, 1):
        p = dict(convergence_residue=1e-9, max_iterations=3 * restart + 2, preconditioner=pre, gmres_variant="CWY",
                 restarting_min=restart, restarting_max=restart)
        ref = O.solve("gmres", rp, c[o].astype(np.int32), v[o], b, **{**p, "gmres_variant": 4})
        ok, its, _, h, x = _run_device_solver(tnl, dev, "gmres", rp, c[o].astype(np.int32), v[o], b, fmt="SlicedEllpack",
                                              **p)
        m = min(len(h), len(ref["history"]), 2 * restart + 2)
        assert abs(len(h) - len(ref["history"])) <= 1 and abs(its - ref["iterations"]) <= 1
        # Householder vectors keep the basis orthogonal to rounding: the sums' order shows at 1e-13 a step
        np.testing.assert_allclose(h[:m], ref["history"][:m], rtol=1e-8, atol=1e-13)


@pytest.mark.parametrize("fmt", ["CSRScalar", "CSRAdaptive", "Ellpack", "SlicedEllpack", "ChunkedEllpack", "BiEllpack"])
@pytest.mark.parametrize("dt,degree", [("f64", 0), ("f64", 1), ("f64", 2), ("f32", 3)])
def test_polynomial_start_in_the_product_of_every_format(tnl, dev, fmt, dt, degree):
    # z_0 = D^-1 A v stored beside the product: every format's run follows the CSRScalar one
    rp, c, v = W.convection_diffusion_3d(9, 10.0)
    b = W.uniform_vector(len(rp) - 1, 4)
    p = dict(dtype=dt, convergence_residue=1e-9 if dt == "f64" else 1e-4, max_iterations=200, preconditioner=3,
             poly_degree=degree, restarting_min=10, restarting_max=10)
    want = _run_device_solver(tnl, dev, "gmres", rp, c, v, b, fmt="CSRScalar", **p)
    got = _run_device_solver(tnl, dev, "gmres", rp, c, v, b, fmt=fmt, **p)
    assert got[0] and want[0] and abs(got[1] - want[1]) <= 1
    np.testing.assert_allclose(got[3][:8], want[3][:8], rtol=1e-9 if dt == "f64" else 1e-3)


def test_polynomial_over_a_striped_plan(tnl, dev):
    # a striped plan forms z_0 in a pass of its own; its row sums differ from the plain product's by
    # their order alone
    rp, c, v = W.convection_diffusion_3d(9, 10.0)
    b = t(W.uniform_vector(len(rp) - 1, 4), dev)
    h = []
    for stripes in (0, 4):
        A = tnl.SparseMatrix.from_csr(rp, c, v, format="CSRAdaptive", dtype="f64")
        A.set_param("column_stripes", stripes)
        s = tnl.getLinearSolver("gmres")
        s.setMatrix(A)
        s.setup(convergence_residue=1e-9, max_iterations=200, preconditioner=3, restarting_min=10, restarting_max=10)
        assert s.solve(b, torch.zeros_like(b))
        h.append(s.getResidualHistory())
    assert abs(len(h[0]) - len(h[1])) <= 1
    np.testing.assert_allclose(h[0][:8], h[1][:8], rtol=1e-9)


@pytest.mark.parametrize("method", ["cg", "bicgstab"])
@pytest.mark.parametrize("most", [0, 1, 2, 11, 12, 13, 29])
def test_iteration_limits_of_fused_solves(tnl, dev, method, most):
    rp, c, v = W.laplacian_2d(24)
    b = W.uniform_vector(len(rp) - 1, 5)
    p = dict(convergence_residue=1e-30, max_iterations=most)
    ref = O.solve(method, rp, c, v, b, **p)
    ok, its, _, h, x = _run_device_solver(tnl, dev, method, rp, c, v, b, fmt="SlicedEllpack", **p)
    assert not ok and its == ref["iterations"] and len(h) == len(ref["history"])
    np.testing.assert_allclose(x, ref["x"], rtol=0, atol=1e-7 * np.abs(ref["x"]).max() + 1e-300)


def _solve_us(tnl, dev, method, dtype, most, repeats):
    """Shortest time of a solve cut off after `most` iterations, and the iterations it made; diagonally dominant, so that
    FP32 is at its rounding level within tens of iterations."""
    rp, c, v = W.laplacian_2d(205)
    v = np.where(v > 0, 6.5, v)
    A = tnl.SparseMatrix.from_csr(rp, c, v, format="SlicedEllpack", dtype=dtype)
    s = tnl.getLinearSolver(method)
    s.setMatrix(A)
    s.setup(convergence_residue=1e-300, max_iterations=most)
    b = t(W.uniform_vector(len(rp) - 1, 3), dev, A.vector_dtype)
    best = 1e9
    for _ in range(repeats):
        x = torch.zeros_like(b)
        torch.cuda.synchronize()
        start = time.perf_counter()
        s.solve(b, x)
        best = min(best, 1e6 * (time.perf_counter() - start))
    return best, s.getIterations()


@pytest.mark.parametrize("method", ["cg", "bicgstab"])
def test_a_solve_of_the_eager_batches_builds_no_graph(tnl, dev, method):
    """The launches that close the last of 4 and 8 iterations belong to the eager batches: cut off after 11 (one more is
    counted) a solve costs about 1.05 times the 10, with a graph built for the closing launches 1.6 times."""
    ten, eleven = (_solve_us(tnl, dev, method, "f64", most, 20)[0] for most in (10, 11))
    assert eleven < 1.3 * ten, (ten, eleven)


def test_launches_behind_the_stop_leave_the_matrix_alone(tnl, dev):
    """A CG solve cut off after 13 iterations replays 16, most of them behind the stop: 1.49 times the 10 that need no
    replay; with the closed products' first rows loaded all the same 1.79 times."""
    rp, c, v = W.laplacian_3d(150)
    A = tnl.SparseMatrix.from_csr(rp, c, v, format="SlicedEllpack", dtype="f64")
    b = t(W.uniform_vector(len(rp) - 1, 3), dev)
    s = tnl.getLinearSolver("cg")
    s.setMatrix(A)
    took = {}
    for most in (10, 13):
        s.setup(convergence_residue=1e-300, max_iterations=most)
        for _ in range(12):
            x = torch.zeros_like(b)
            torch.cuda.synchronize()
            start = time.perf_counter()
            s.solve(b, x)
            took[most] = min(took.get(most, 1e9), time.perf_counter() - start)
    assert took[13] < 1.7 * took[10], took


@pytest.mark.parametrize("method,vectors", [("cg", 4), ("bicgstab", 7)])
def test_large_solves_keep_one_set_of_vectors(tnl, dev, method, vectors):
    """Beyond the rows whose operands the products form, a solve allocates what it did with separate passes."""
    rp, c, v = W.laplacian_2d(2000)
    A = tnl.SparseMatrix.from_csr(rp, c, v, format="SlicedEllpack", dtype="f64")
    s = tnl.getLinearSolver(method)
    s.setMatrix(A)
    s.setup(convergence_residue=1e-300, max_iterations=2)
    b = t(W.uniform_vector(len(rp) - 1, 3), dev)
    x = torch.zeros_like(b)
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    s.solve(b, x)
    used = before - torch.cuda.mem_get_info()[0]
    size = 8 * (len(rp) - 1)
    assert used < (vectors + 0.9) * size, used / size


def test_restarts_do_not_queue_ahead_of_each_other(tnl, dev):
    """FP32 BiCGStab that cannot get any lower restarts again and again; an iteration then costs 1.1 times one of
    the FP64 solve, which does not (1.36 times with up to 64 iterations queued behind every restart)."""
    (low, its), (high, n) = (_solve_us(tnl, dev, "bicgstab", d, 1000, 4) for d in ("f32", "f64"))
    assert its >= 1000 and n >= 1000
    assert low / its < 1.24 * high / n, (low / its, high / n)


@pytest.mark.parametrize("fmt", ["SlicedEllpack", "CSRAdaptive"])
def test_ilu0_wide_levels_follow_the_oracle(tnl, dev, fmt):
    """ILU(0) on the 64^3 Laplacian: the anti-diagonal planes hold up to 3072 rows, so the
    schedule mixes one-workgroup runs of small levels with device-wide levels.  CG follows the
    oracle's (TNL's) history and iteration count; BiCGStab, whose iteration count moves with the
    rounding of its dot products, follows the history of its first iterations."""
    rp, c, v = W.laplacian_3d(64)
    b = W.uniform_vector(len(rp) - 1, 5)
    kw = dict(convergence_residue=1e-8, max_iterations=500, preconditioner=2)
    for method, first in (("cg", 30), ("bicgstab", 10)):
        ref = O.solve(method, rp, c, v, b, **kw)
        ok, its, res, hist, x = _run_device_solver(tnl, dev, method, rp, c, v, b, fmt=fmt, **kw)
        print(method, its, ref["iterations"], hist[:first], ref["history"][:first], flush=True)
        assert ok and ref["converged"], method
        if method == "cg":
            assert abs(its - ref["iterations"]) <= 2, (its, ref["iterations"])
        np.testing.assert_allclose(hist[:first], ref["history"][:first], rtol=1e-6, err_msg=method)
        r = b - _csr_matvec(rp, c, v, x)
        assert np.linalg.norm(r) / np.linalg.norm(b) < 5e-8, method
    ok32, its32, res32, _, _ = _run_device_solver(tnl, dev, "bicgstab", rp, c, v, b, fmt=fmt, dtype="f32",
                                                  convergence_residue=1e-5, max_iterations=500, preconditioner=2)
    assert ok32 and its32 <= its + 5


def _ilu_matrix(kind):
    """Matrices whose triangular sweeps take each path of the device schedule."""
    rng = np.random.default_rng(17)
    if kind == "chain":  # every level one row, an odd number of them
        n, per = 1501, [np.array([i - 1]) if i else np.array([], int) for i in range(1501)]
    elif kind == "long rows":  # more entries than are fetched ahead, mixed lengths in a level
        n = 4000
        per = [np.unique(rng.integers(max(0, i - 900), max(i, 1), rng.integers(0, 12) if i % 7 else 40)) for i in range(n)]
    elif kind == "far columns":  # dependencies older than the 16384 solution entries kept in LDS
        n = 45000
        per = [np.unique(np.concatenate([[i - 1500], rng.integers(0, i - 1500, 2)])) if i > 1500 else np.array([], int)
               for i in range(n)]
    else:  # levels on both sides of 4096 rows, or of the 1024 from which far columns make a launch of a level
        sizes = ([4096, 4097, 3, 1, 1025, 6000, 4095, 64] if kind == "wide levels" else
                 [4000] * 4 + [3000, 1024, 1025, 2, 130, 1026, 1500, 1000, 2000])
        start = np.concatenate([[0], np.cumsum(sizes)])
        n, per = int(start[-1]), []
        for lv, size in enumerate(sizes):
            for k in range(size):
                per.append(np.array([], int) if lv == 0 else np.unique(
                    np.concatenate([rng.integers(start[lv - 1], start[lv], 1), rng.integers(0, start[lv], 2)])))
    rows, cols, vals = [], [], []
    for i in range(n):
        low = per[i][per[i] < i]
        up = [j for j in range(i + 1, min(n, i + 1 + i % 5))]
        c = np.concatenate([low, [i] * (2 if i % 11 == 3 else 1), up]).astype(np.int32)
        v = rng.uniform(-1, 1, len(c))
        v[c == i] = 2.0 + len(c) / (2 if i % 11 == 3 else 1)
        rows.append(len(c))
        cols.append(c)
        vals.append(v)
    rp = np.concatenate([[0], np.cumsum(rows)]).astype(np.int32)
    return rp, np.concatenate(cols), np.concatenate(vals)


@pytest.mark.parametrize("kind", ["chain", "long rows", "far columns", "wide levels", "far levels"])
def test_ilu0_sweep_paths_follow_the_oracle(tnl, dev, kind):
    """The triangular sweeps give TNL's bits on every path (rows longer than the fetched entries, a
    second entry on the diagonal, columns older than the LDS ring, one-row and device-wide levels),
    so the first residuals differ by the rounding of the solver's dot products only: sums of 45,000
    terms in another order, about 1e-13 relative, a few of them per iteration."""
    rp, c, v = _ilu_matrix(kind)
    b = W.uniform_vector(len(rp) - 1, 5)
    kw = dict(convergence_residue=1e-30, max_iterations=3, preconditioner=2)
    ref = O.solve("bicgstab", rp, c, v, b, **kw)
    _, _, _, hist, _ = _run_device_solver(tnl, dev, "bicgstab", rp, c, v, b, fmt="CSRScalar", **kw)
    print(kind, hist[:4], ref["history"][:4], flush=True)
    np.testing.assert_allclose(hist[:3], ref["history"][:3], rtol=1e-9)
    _, _, _, h32, _ = _run_device_solver(tnl, dev, "bicgstab", rp, c, v, b, fmt="CSRScalar", dtype="f32", **kw)
    np.testing.assert_allclose(h32[:2], ref["history"][:2], rtol=2e-3)  # FP32 factors and vectors


def _levelled(levels, per, entries):
    """`levels` levels of `per` rows in both sweeps, each row with `entries` columns anywhere in the levels before."""
    rng = np.random.default_rng(2)
    n = levels * per
    i = np.arange(per, n)
    low = (rng.random((len(i), entries)) * (i // per * per)[:, None]).astype(np.int64)
    low[:, 0] = i - per
    r = np.concatenate([np.arange(n), np.repeat(i, entries), i - per])
    c = np.concatenate([np.arange(n), low.ravel(), i])
    key, first = np.unique(r * n + c, return_index=True)
    v = np.concatenate([np.full(n, 2.0 * entries), rng.uniform(-1, 1, low.size + len(i))])[first]
    rp = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(key // n, minlength=n), out=rp[1:])
    return rp, (key % n).astype(np.int32), v


def _ilu_ms_per_level(tnl, dev, m, levels):
    rp, c, v = m
    b = t(W.uniform_vector(len(rp) - 1, 3), dev)
    s = tnl.getLinearSolver("bicgstab")
    s.setMatrix(tnl.SparseMatrix.from_csr(rp, c, v, format="CSRAdaptive", dtype="f64"))
    s.setup(convergence_residue=1e-300, max_iterations=4, preconditioner=2)
    best = 1e9
    for _ in range(3):  # the first one builds the factors
        x = torch.zeros_like(b)
        torch.cuda.synchronize()
        start = time.perf_counter()
        s.solve(b, x)
        best = min(best, 1e3 * (time.perf_counter() - start))
    return best / levels


def test_ilu0_sweep_cost_follows_the_levels(tnl, dev):
    """What a level of a triangular sweep costs: a level of one row a fraction of one of 1400 (a run's workgroup is as
    large as its levels; 0.3 measured, 0.8 with 16 waves for every run), and 2500 rows whose columns lie anywhere before
    them no more than 6000 such rows, which are a launch (0.9 measured, 2.6 in a run)."""
    n = 4000
    i = np.arange(n)
    r, c = np.concatenate([i[1:], i, i[:-1]]), np.concatenate([i[1:] - 1, i, i[:-1] + 1])
    o = np.lexsort((c, r))
    rp = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(r, minlength=n), out=rp[1:])
    chain = _ilu_ms_per_level(tnl, dev, (rp, c[o].astype(np.int32), np.where(c == r, 4.0, -1.0)[o]), n)
    grid = _ilu_ms_per_level(tnl, dev, W.laplacian_3d(64), 190)
    assert chain < 0.5 * grid, (chain, grid)
    few, many = (_ilu_ms_per_level(tnl, dev, _levelled(40, rows, 13), 40) for rows in (2500, 6000))
    assert few < 1.6 * many, (few, many)


def test_ilu0_refuses_rows_without_an_upper_entry(tnl, dev):
    # row 2 holds only a column below the diagonal: no U_22 to divide by
    rp = np.array([0, 1, 2, 3], np.int32)
    c = np.array([0, 1, 0], np.int32)
    v = np.array([2.0, 3.0, 1.0])
    with pytest.raises(tnl.TnlHipError, match="no entry on or above the diagonal"):
        _run_device_solver(tnl, dev, "cg", rp, c, v, np.ones(3), preconditioner=2)


def _csr_matvec(rp, c, v, x):
    rows = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
    return np.bincount(rows, weights=v * x[c], minlength=len(rp) - 1)


def test_symmetric_matrix_solves(tnl, dev):
    """CG (plain and with Jacobi) on a SymmetricMatrix holding the lower triangle of the 3-D
    Laplacian follows the oracle's CG on the full matrix; ILU(0) refuses the symmetric type."""
    rp, c, v = W.laplacian_3d(16)
    n = len(rp) - 1
    rows = np.repeat(np.arange(n), np.diff(rp))
    keep = c <= rows
    lrp = np.concatenate([[0], np.cumsum(np.bincount(rows[keep], minlength=n))]).astype(np.int32)
    b = W.uniform_vector(n, 9)
    for pre in (0, 1):
        ref = O.solve("cg", rp, c, v, b, convergence_residue=1e-10, max_iterations=2000, preconditioner=pre)
        A = tnl.SparseMatrix.symmetric_from_csr(lrp, c[keep], v[keep], format="SlicedEllpack")
        s = tnl.getLinearSolver("cg")
        s.setMatrix(A)
        s.setup(convergence_residue=1e-10, max_iterations=2000, preconditioner=pre)
        x = torch.zeros(n, dtype=torch.float64, device=dev)
        assert s.solve(t(b, dev, torch.float64), x)
        assert abs(s.getIterations() - ref["iterations"]) <= 2, (pre, s.getIterations(), ref["iterations"])
        np.testing.assert_allclose(s.getResidualHistory()[:30], ref["history"][:30], rtol=1e-6)
    s = tnl.getLinearSolver("cg")
    s.setMatrix(A)
    s.setup(preconditioner=2)
    with pytest.raises(tnl.TnlHipError, match="symmetric"):
        s.solve(t(b, dev, torch.float64), torch.zeros(n, dtype=torch.float64, device=dev))


def _parse_history(text):
    """(iteration, residue) lines and the positions of the blank lines of a residual history file."""
    rows, blanks = [], []
    for line in text.split("\n"):
        if line == "":
            blanks.append(len(rows))
            continue
        it, r = line.split("\t")
        rows.append((int(it), float(r)))
    return rows, blanks


def test_residual_history_file_and_monitor_follow_tnl(tnl, dev, tmp_path):
    """setup( residual-history-file ) and setSolverMonitor: the file TNL writes
    (IterativeSolver.hpp:189-200: a blank line at iteration 0, then "<iteration>\\t<residue>"),
    compared with TNL's own file for the same solve -- iteration numbers equal line by line over the
    first lines, residues within the device's rounding -- and a monitor that last sees the final
    (iterations, residue)."""
    hist = np.load(os.path.join(ROOT, "tests", "golden", "history.npz"))
    sol = np.load(os.path.join(ROOT, "tests", "golden", "solvers.npz"))
    runs = sorted({k.split("/")[0] for k in hist.files})
    for run in runs:
        sysname, method = str(hist[f"{run}/system"]), str(hist[f"{run}/method"])
        params = dict(eval(str(hist[f"{run}/params"])))
        print(f"history {run} {sysname} {method} {params}", flush=True)
        rp, c, v, b = (sol[f"{sysname}/{k}"] for k in ("row_ptr", "cols", "vals", "b"))
        A = tnl.SparseMatrix.from_csr(rp, c, v, format="CSRScalar", dtype="f64")
        s = tnl.getLinearSolver(method)
        s.setMatrix(A)
        s.setup(**params)
        path = tmp_path / f"{run}.txt"
        s.setResidualHistoryFile(path)
        seen = []
        s.setSolverMonitor(lambda it, r: seen.append((it, r)))
        x = torch.zeros(len(b), dtype=torch.float64, device=dev)
        s.solve(torch.tensor(b, device=dev), x)
        s.setResidualHistoryFile(None)  # closes the file
        ours, ours_blank = _parse_history(path.read_text())
        ref, ref_blank = _parse_history(str(hist[f"{run}/text"]))
        assert ours_blank[0] == 0 and ref_blank[0] == 0, run
        m = min(len(ours), len(ref), 20)
        assert [i for i, _ in ours[:m]] == [i for i, _ in ref[:m]], run
        np.testing.assert_allclose([r for _, r in ours[:m]], [r for _, r in ref[:m]], rtol=2e-6, atol=1e-14,
                                   err_msg=run)
        assert [i for i, _ in ours] == list(s.getResidualHistoryIterations()), run
        np.testing.assert_allclose([r for _, r in ours], s.getResidualHistory(), rtol=1e-6, err_msg=run)
        assert seen and seen[-1] == (s.getIterations(), s.getResidue()), run
