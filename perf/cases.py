"""The sparse-matrix work of a program that uses this framework, as cases that can be timed and checked.

Five kinds of call cover the path from one matrix-vector product to a solve service:

  spmv    SparseMatrix.vectorProduct              y = alpha A x + beta y
  multi   SparseMatrix.vectorProductMulti         the same for a row-major block of k vectors
  solve   CG / BICGStab / GMRES .solve            A x = b from x = 0 to a relative residual
  refine  refine_solve                            FP64 refinement over an FP32 solve
  serve   Server.submit / run_all                 many shifted systems at once, host arrays in and out

Matrices are the 5- and 7-point Laplacians, the upwind convection-diffusion operator and the
irregular matrix (lognormal row lengths, columns anywhere) of the package's workloads module,
assembled here on the GPU so that inputs are quick to make; boxes need not be cubes.
"""
import importlib
import math

import numpy as np
import torch

tnl = importlib.import_module("tnl-dev_amd")

DEV = "cuda"
FORMATS = ("CSRScalar", "CSRVector", "CSRLight", "CSRHybrid", "CSRAdaptive", "Ellpack", "SlicedEllpack",
           "ChunkedEllpack", "BiEllpack")
VECTOR = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.float32}
STORED = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16}
VALUE_BYTES = {"f64": 8, "f32": 4, "bf16": 2}


# ------------------------------------------------------------------ the cases


def listed():
    return [
        # the smallest product: a 2D grid that TNL's own users run on the host, one launch of a
        # few microseconds; what it costs is what every step of a small time-stepping loop costs
        {"name": "spmv-2d-256", "kind": "spmv", "matrix": "laplacian", "nx": 256, "ny": 256, "nz": 1,
         "format": "CSRScalar", "dtype": "f64", "alpha": 1.0, "beta": 0.0},
        # the benchmark's headline product: a 3D grid whose matrix streams from HBM
        {"name": "spmv-3d-160", "kind": "spmv", "matrix": "laplacian", "nx": 160, "ny": 160, "nz": 160,
         "format": "ChunkedEllpack", "dtype": "f64", "alpha": 1.0, "beta": 0.0},
        # single precision with an update of y (alpha A x + beta y) on an odd, non-cubic box
        {"name": "spmv-3d-f32-update", "kind": "spmv", "matrix": "convection", "nx": 127, "ny": 150, "nz": 93,
         "peclet": 10.0, "format": "SlicedEllpack", "dtype": "f32", "alpha": -1.0, "beta": 1.0},
        # rows of very different lengths with columns anywhere (graphs, circuits): the benchmark's
        # irregular matrix in the format made for such rows
        {"name": "spmv-irregular-2m", "kind": "spmv", "matrix": "irregular", "rows": 2000000, "mean": 16.0,
         "sigma": 1.2, "format": "CSRAdaptive", "dtype": "f64", "alpha": 1.0, "beta": 0.0},
        # a block of right-hand sides (block Krylov methods, many load cases)
        {"name": "multi-3d-k16", "kind": "multi", "matrix": "laplacian", "nx": 128, "ny": 128, "nz": 128, "k": 16,
         "format": "SlicedEllpack", "dtype": "f64", "alpha": 1.0, "beta": 0.0},
        # a small Poisson problem: hundreds of short iterations, so launches and latency count
        {"name": "cg-2d-256", "kind": "solve", "method": "cg", "matrix": "laplacian", "nx": 256, "ny": 256, "nz": 1,
         "format": "CSRScalar", "preconditioner": 0, "residue": 1e-8},
        # a large Poisson problem with the Jacobi preconditioner: bandwidth counts
        {"name": "cg-3d-128-jacobi", "kind": "solve", "method": "cg", "matrix": "laplacian", "nx": 128, "ny": 128,
         "nz": 128, "format": "SlicedEllpack", "preconditioner": 1, "residue": 1e-8},
        # convection-diffusion (nonsymmetric) with BiCGStab, the usual first choice for it
        {"name": "bicgstab-3d-64-jacobi", "kind": "solve", "method": "bicgstab", "matrix": "convection", "nx": 64,
         "ny": 64, "nz": 64, "peclet": 10.0, "format": "SlicedEllpack", "preconditioner": 1, "residue": 1e-10},
        # the same system with ILU(0), whose triangular solves are a chain of dependent levels
        {"name": "bicgstab-3d-64-ilu0", "kind": "solve", "method": "bicgstab", "matrix": "convection", "nx": 64,
         "ny": 64, "nz": 64, "peclet": 10.0, "format": "SlicedEllpack", "preconditioner": 2, "residue": 1e-10},
        # restarted GMRES with the default (Householder) orthogonalization at the benchmark's size
        {"name": "gmres-3d-128-cwy", "kind": "solve", "method": "gmres", "variant": "CWY", "restart": 30,
         "matrix": "convection", "nx": 128, "ny": 128, "nz": 128, "peclet": 100.0, "format": "CSRAdaptive",
         "preconditioner": 1, "residue": 1e-10},
        # FP64 accuracy from FP32 GMRES with the BF16 Jacobi-polynomial preconditioner
        {"name": "refine-3d-128", "kind": "refine", "matrix": "convection", "nx": 128, "ny": 128, "nz": 128,
         "peclet": 10.0, "format": "SlicedEllpack", "residue": 1e-10},
        # a burst at the solve service: 32 requests of mixed sizes, one in five of them GMRES
        {"name": "serve-32", "kind": "serve", "requests": 32, "most_rows": 250000, "gmres_every": 5,
         "residue": 1e-10},
    ]


def _box(rng, low, high):
    """Sides of a 2D or 3D box with about log-uniform many rows in [low, high]; odd sizes among them."""
    n = math.exp(rng.uniform(math.log(low), math.log(high)))
    d = 2 if rng.random() < 0.35 else 3
    s = [n ** (1.0 / d) * math.exp(rng.uniform(-0.25, 0.25)) for _ in range(d - 1)]
    s.append(n / math.prod(s))
    s = [max(8, int(v)) for v in s] + [1] * (3 - d)
    while math.prod(s) > high:
        s[s.index(max(s))] -= 1
    return {"nx": s[0], "ny": s[1], "nz": s[2]}


def draw(rng):
    kind = rng.choice(("spmv",) * 5 + ("multi",) * 2 + ("solve",) * 5 + ("refine", "serve"))
    if kind == "spmv":
        dtype = rng.choice(("f64", "f64", "f32", "bf16"))
        case = {"kind": kind, "format": rng.choice(FORMATS), "dtype": dtype,
                "alpha": rng.choice((1.0, 1.0, 0.75, -1.0)), "beta": rng.choice((0.0, 0.0, 0.5, 1.0))}
        if rng.random() < 0.3:
            case.update(matrix="irregular", rows=int(math.exp(rng.uniform(math.log(2e4), math.log(2e6)))),
                        mean=rng.choice((8.0, 16.0)), sigma=rng.choice((0.6, 1.2)))
            if case["format"] == "Ellpack":  # would store every row at the longest one's length
                case["format"] = "CSRAdaptive"
        else:
            case.update(matrix=rng.choice(("laplacian", "convection")), **_box(rng, 4e3, 4.0e6))
    elif kind == "multi":
        case = {"kind": kind, "matrix": rng.choice(("laplacian", "convection")), "k": rng.choice((2, 3, 4, 7, 8, 12, 16)),
                "format": rng.choice(FORMATS), "dtype": rng.choice(("f64", "f64", "f32")), "alpha": 1.0,
                "beta": rng.choice((0.0, 1.0)), **_box(rng, 4e3, 2.0e6)}
    elif kind == "solve":
        method = rng.choice(("cg", "cg", "bicgstab", "gmres"))
        pre = rng.choice((0, 1, 1, 2))
        case = {"kind": kind, "method": method, "preconditioner": pre, "residue": rng.choice((1e-8, 1e-10)),
                "matrix": "laplacian" if method == "cg" else "convection",
                "format": rng.choice(("CSRScalar", "CSRAdaptive", "Ellpack", "SlicedEllpack", "ChunkedEllpack",
                                      "BiEllpack")), **_box(rng, 4e3, 2.5e5 if pre == 2 else 1.5e6)}
        if pre == 2:  # the ILU(0) of a 3D box (a 2D one has far more levels to a row)
            while case["nz"] == 1:
                case.update(_box(rng, 4e3, 2.5e5))
        if method == "gmres":
            case.update(variant=rng.choice(("CWY", "CWY", "CGS", "CGSR", "MGS")), restart=rng.choice((10, 20, 30)))
            while case["nz"] == 1:  # restarted GMRES is for the 3D box here
                case.update(_box(rng, 4e3, 2.5e5 if pre == 2 else 1.0e6))
    elif kind == "refine":
        case = {"kind": kind, "matrix": "convection", "format": rng.choice(("CSRAdaptive", "SlicedEllpack",
                                                                            "ChunkedEllpack")),
                "residue": 1e-10, **_box(rng, 3e4, 2.0e6)}
        while case["nz"] == 1:
            case.update(_box(rng, 3e4, 2.0e6))
    else:
        case = {"kind": kind, "requests": rng.randint(6, 32), "most_rows": rng.choice((60000, 120000, 250000)),
                "gmres_every": rng.choice((0, 3, 5)), "residue": 1e-10}
    if case.get("matrix") == "convection":
        case["peclet"] = rng.choice((10.0, 30.0, 100.0))
    return case


# ------------------------------------------------------------------ matrices (device CSR)


def _stencil(nx, ny, nz, entries):
    """Device CSR of a constant-coefficient stencil on an nx x ny x nz box (x fastest, Dirichlet
    truncation); entries: ((dx, dy, dz), value) in ascending order of the linear offset."""
    n = nx * ny * nz
    i = torch.arange(n, device=DEV)
    x, y, z = i % nx, (i // nx) % ny, i // (nx * ny)
    cols, on, vals = [], [], []
    for (dx, dy, dz), v in entries:
        on.append((x + dx >= 0) & (x + dx < nx) & (y + dy >= 0) & (y + dy < ny) & (z + dz >= 0) & (z + dz < nz))
        cols.append(i + dx + nx * dy + nx * ny * dz)
        vals.append(v)
    on = torch.stack(on, 1)
    rp = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(on.sum(1), 0, out=rp[1:])
    cols = torch.stack(cols, 1)[on].to(torch.int32)
    vals = torch.tensor(vals, dtype=torch.float64, device=DEV).expand(n, len(entries))[on]
    return rp.to(torch.int32), cols, vals.contiguous()


def _laplacian(nx, ny, nz):
    e = [((0, -1, 0), -1.0), ((-1, 0, 0), -1.0), ((0, 0, 0), 4.0 if nz == 1 else 6.0), ((1, 0, 0), -1.0),
         ((0, 1, 0), -1.0)]
    if nz > 1:
        e = [((0, 0, -1), -1.0)] + e + [((0, 0, 1), -1.0)]
    return _stencil(nx, ny, nz, e)


def _convection(nx, ny, nz, peclet):
    """-Laplace(u) + Pe (1, 0.5, 0.25) . grad u, first-order upwind, rows scaled by h^2."""
    h = 1.0 / (max(nx, ny, nz) + 1)
    vx, vy, vz = peclet * h, 0.5 * peclet * h, (0.25 * peclet * h if nz > 1 else 0.0)
    e = [((0, -1, 0), -1.0 - vy), ((-1, 0, 0), -1.0 - vx), ((0, 0, 0), (4.0 if nz == 1 else 6.0) + vx + vy + vz),
         ((1, 0, 0), -1.0), ((0, 1, 0), -1.0)]
    if nz > 1:
        e = [((0, 0, -1), -1.0 - vz)] + e + [((0, 0, 1), -1.0)]
    return _stencil(nx, ny, nz, e)


def _irregular(n, mean, sigma, seed):
    """Off-diagonal row lengths lognormal (the given mean) in [1, 4096], columns uniform, values
    U[-1, 1], diagonal 1 + the row's length (diagonally dominant)."""
    g = torch.Generator(device=DEV).manual_seed(seed * 7 + 3)
    mu = math.log(mean) - sigma * sigma / 2.0
    z = torch.randn(n, generator=g, device=DEV, dtype=torch.float64)
    length = torch.exp(mu + sigma * z).round().clamp(1, min(4096, n - 1)).to(torch.int64)
    rows = torch.repeat_interleave(torch.arange(n, device=DEV), length)
    key = rows * n + torch.randint(0, n, (rows.numel(),), generator=g, device=DEV)
    key = torch.unique(torch.cat([key, torch.arange(n, device=DEV) * (n + 1)]))  # sorted, repeats dropped
    rows, cols = key // n, key % n
    vals = torch.rand(key.numel(), generator=g, device=DEV, dtype=torch.float64) * 2 - 1
    count = torch.bincount(rows, minlength=n)
    vals = torch.where(rows == cols, 1.0 + count[rows].to(torch.float64), vals)
    rp = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    torch.cumsum(count, 0, out=rp[1:])
    return rp.to(torch.int32), cols.to(torch.int32), vals


def _csr(case, seed):
    if case["matrix"] == "irregular":
        return _irregular(case["rows"], case["mean"], case["sigma"], seed)
    if case["matrix"] == "laplacian":
        return _laplacian(case["nx"], case["ny"], case["nz"])
    return _convection(case["nx"], case["ny"], case["nz"], case["peclet"])


def _matrix(case, csr, dtype):
    return tnl.SparseMatrix.from_csr(*csr, format=case["format"], dtype=dtype)


def _product(csr, x):
    """A x in FP64 by plain torch; x is a vector or a block of columns."""
    rp, cols, vals = csr
    lengths = (rp[1:] - rp[:-1]).to(torch.int64)
    if x.dim() == 1:
        return torch.segment_reduce(vals * x[cols], "sum", lengths=lengths, unsafe=True)
    return torch.stack([_product(csr, x[:, j].contiguous()) for j in range(x.shape[1])], 1)


# ------------------------------------------------------------------ inputs


def _uniform(shape, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    return torch.rand(shape, generator=g, device=DEV, dtype=torch.float64) * 2 - 1


def _solution(nx, ny, nz, seed, columns=1):
    """A solution field as a discretized problem has it: a few smooth modes with random
    coefficients, and 1 % of noise; (rows, columns)."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    out = []
    for _ in range(columns):
        f = 0.01 * (torch.rand(nx * ny * nz, generator=g, device=DEV, dtype=torch.float64) * 2 - 1).view(nz, ny, nx)
        for _ in range(6):
            s = [torch.sin(math.pi * m * (torch.arange(k, device=DEV, dtype=torch.float64) + 1) / (k + 1))
                 for k, m in zip((nz, ny, nx), torch.randint(1, 7, (3,), generator=g, device=DEV).tolist())]
            if nz == 1:
                s[0] = torch.ones(1, dtype=torch.float64, device=DEV)
            c = torch.randn((), generator=g, device=DEV, dtype=torch.float64)
            f = f + c * s[0][:, None, None] * s[1][None, :, None] * s[2][None, None, :]
        out.append(f.reshape(-1))
    return torch.stack(out, 1)


# Resident matrices of the service: grid sides of 2D and 3D Laplacians from a thousand rows up.
LADDER = ((32, 32, 1), (89, 89, 1), (199, 199, 1), (345, 345, 1), (500, 500, 1),
          (10, 10, 10), (22, 22, 22), (36, 36, 36), (49, 49, 49), (62, 62, 62))


def _requests(case, seed):
    """(box, shift, right-hand sides, method, seed) of each request; the boxes, shifts and counts are the
    case's own, so that the work does not change with the seed."""
    rng = np.random.default_rng(case["requests"] * 1000 + case["most_rows"] % 997)
    sides = [s for s in LADDER if math.prod(s) <= case["most_rows"]]
    out = []
    for q in range(case["requests"]):
        box = sides[int(rng.integers(len(sides)))]
        every = case["gmres_every"]
        out.append((box, float(rng.uniform(0.02, 1.0)), int(rng.integers(1, 17)),
                    "gmres" if every and q % every == every - 1 else "cg", seed * 1000 + q))
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "serve":
        return _prepare_serve(case, seed)
    csr = _csr(case, seed)
    n = csr[0].numel() - 1
    if kind in ("spmv", "multi"):
        dt = VECTOR[case["dtype"]]
        shape = (n,) if kind == "spmv" else (n, case["k"])
        return {"case": case, "A": _matrix(case, csr, case["dtype"]), "x": _uniform(shape, seed).to(dt),
                "y": _uniform(shape, seed + 500009).to(dt)}
    x = _solution(case["nx"], case["ny"], case["nz"], seed)[:, 0].contiguous()
    state = {"case": case, "A": _matrix(case, csr, "f64"), "b": _product(csr, x), "x": torch.zeros_like(x)}
    if kind == "refine":
        state["low"] = _matrix(case, csr, "f32")
        state["poly"] = _matrix(case, csr, "bf16")
        state["context"] = tnl.RefineContext()
        return state
    s = tnl.getLinearSolver(case["method"])
    s.setMatrix(state["A"])
    s.setup(convergence_residue=case["residue"], max_iterations=100000, preconditioner=case["preconditioner"])
    if case["method"] == "gmres":
        s.setup(restarting_min=case["restart"], restarting_max=case["restart"], gmres_variant=case["variant"])
    state["solver"] = s
    return state


def _prepare_serve(case, seed):
    reqs = _requests(case, seed)
    boxes = sorted({r[0] for r in reqs})
    csrs = {b: _laplacian(*b) for b in boxes}
    slots = sum(7 * math.prod(b) + 4096 for b in boxes) * 2
    entries = sum(math.prod(r[0]) * (r[2] + 1) + 4096 for r in reqs)
    server = tnl.Server(vector_capacity=entries, matrix_capacity=slots,
                        slice_capacity=sum(math.prod(b) // 32 + 64 for b in boxes), max_requests=64)
    ids = {b: server.add_matrix(*[t.cpu().numpy() for t in csrs[b]]) for b in boxes}
    work = []
    for box, shift, k, method, s in reqs:
        x = _solution(*box, s, k)
        work.append((ids[box], (_product(csrs[box], x) + shift * x).cpu().numpy(), shift, method))
    return {"case": case, "server": server, "work": work}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "spmv":
        return state["A"].vectorProduct(state["x"], state["y"], case["alpha"], case["beta"])
    if kind == "multi":
        return state["A"].vectorProductMulti(state["x"], state["y"], case["alpha"], case["beta"])
    if kind == "solve":
        state["x"].zero_()
        state["solver"].solve(state["b"], state["x"])
        return state["x"]
    if kind == "refine":
        state["x"].zero_()
        tnl.refine_solve(state["A"], state["b"], state["x"], A_low=state["low"], P=state["poly"],
                         tolerance=case["residue"], inner_method="gmres", inner_dtype="f32",
                         convergence_residue=1e-2, max_iterations=3000, restarting_min=30, restarting_max=30,
                         preconditioner=3, poly_degree=3, context=state["context"])
        return state["x"]
    server = state["server"]
    # GMRES requests refine over restarted GMRES, which a loose inner target suits best
    tickets = [server.submit(i, B, shift=shift, tolerance=case["residue"],
                             inner_tolerance=3e-6 if method == "cg" else 1e-2, method=method)
               for i, B, shift, method in state["work"]]
    done = server.run_all()
    return [done[t][0] for t in tickets]


# ------------------------------------------------------------------ work, tolerance, exact values


def _rows_and_entries(case):
    if case["matrix"] == "irregular":
        return case["rows"], int(case["rows"] * (case["mean"] + 1))
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    n = nx * ny * nz
    nnz = n + 2 * (n - ny * nz) + 2 * (n - nx * nz) + (2 * (n - nx * ny) if nz > 1 else 0)
    return n, nnz


def _product_bytes(n, nnz, value_bytes, vector_bytes, k=1, beta=0.0):
    """Values, column indexes and row pointers once, x read and y written once (and read for beta != 0)."""
    return nnz * (value_bytes + 4) + 4 * (n + 1) + k * n * vector_bytes * (3 if beta else 2)


def _iterations(case):
    """About how many iterations the solve takes, from the side of the box and the Peclet number."""
    side = max(case["nx"], case["ny"], case["nz"])
    digits = -math.log10(case["residue"]) / 8.0
    if case["method"] == "cg":
        return side * 2.5 * digits * (0.3 if case["preconditioner"] == 2 else 1.0)
    if case["method"] == "bicgstab":
        return side * 2.4 * digits * (0.3 if case["preconditioner"] == 2 else 1.0)
    return side * 4.4 * digits * (0.3 if case["preconditioner"] == 2 else 1.0)


def work(case):
    """A Krylov step multiplies A with a vector that the step before has made, so a solve reads A and
    its work vectors once for each of its iterations; the products of FP32 and BF16 copies are
    counted at those widths."""
    kind = case["kind"]
    if kind == "serve":
        by = fl = 0.0
        for box, shift, k, _, _ in _requests(case, 0):
            n, nnz = _rows_and_entries({"matrix": "laplacian", "nx": box[0], "ny": box[1], "nz": box[2]})
            cond = (8.0 if box[2] == 1 else 12.0) / shift
            its = 8.0 * math.sqrt(cond)
            by += its * (_product_bytes(n, nnz, 4, 4, k) + 7 * k * n * 4) + 2 * k * n * 8
            fl += its * k * (2 * nnz + 10 * n)
        return {"bytes": by, "flops": fl}
    n, nnz = _rows_and_entries(case)
    if kind in ("spmv", "multi"):
        k = case.get("k", 1)
        return {"bytes": _product_bytes(n, nnz, VALUE_BYTES[case["dtype"]], 8 if case["dtype"] == "f64" else 4, k,
                                        case["beta"]), "flops": 2 * nnz * k}
    if kind == "refine":
        its = 2.5 * max(case["nx"], case["ny"], case["nz"])
        return {"bytes": its * (_product_bytes(n, nnz, 4, 4) + 3 * _product_bytes(n, nnz, 2, 4) + 3 * 15 * n * 4),
                "flops": its * (8 * nnz + 90 * n)}
    its = _iterations(case)
    if case["method"] == "cg":
        per, fl, products = 7 * n * 8, 10 * n, 1
    elif case["method"] == "bicgstab":
        per, fl, products = 14 * n * 8, 20 * n, 2
    else:  # two passes over the basis, half full on average
        per, fl, products = 2 * (case["restart"] / 2) * n * 8, 4 * (case["restart"] / 2) * n, 1
    if case["preconditioner"] == 2:
        per += products * nnz * 12
        fl += products * 2 * nnz
    return {"bytes": its * (products * _product_bytes(n, nnz, 8, 8) + per), "flops": its * (products * 2 * nnz + fl)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("spmv", "multi"):
        # sums of up to 4096 products in another order
        return {"rel": 1e-13, "max": 1e-11} if case["dtype"] == "f64" else {"rel": 2e-6, "max": 1e-4}
    # Two correct solves stop within an iteration or two of each other at the same relative residual;
    # the error that leaves in x was measured against the exact solution: 1.3 (256^2 CG) and 0.5
    # (128^3 CG) times the residual, 5 to 10 (64^3 BiCGStab), 1 (128^3 GMRES), 0.04 to 10
    # (refined solves) over seeds; it grows with the condition number, the square of the side.
    side = 500 if kind == "serve" else max(case["nx"], case["ny"], case["nz"])
    return {"rel": case["residue"] * max(50.0, 8e-5 * side * side)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "serve":
        return [_solution(*box, s, k).cpu().numpy() for box, _, k, _, s in _requests(case, seed)]
    if kind in ("solve", "refine"):
        return _solution(case["nx"], case["ny"], case["nz"], seed)[:, 0]
    rp, cols, vals = _csr(case, seed)
    n = rp.numel() - 1
    shape = (n,) if kind == "spmv" else (n, case["k"])
    dt = VECTOR[case["dtype"]]
    x, y = _uniform(shape, seed).to(dt).double(), _uniform(shape, seed + 500009).to(dt).double()
    r = case["alpha"] * _product((rp, cols, vals.to(STORED[case["dtype"]]).double()), x)
    return r + case["beta"] * y if case["beta"] else r
