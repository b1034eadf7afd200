"""Products with several right-hand sides (tnlhip_spmv_multi) on the GPU: column j of the block
result equals the oracle's one-vector product (TNL's Host order) of column j, bit for bit in FP64,
in every format; keepers, row ranges and the refusals follow tnlhip_spmv."""
import numpy as np
import pytest
import torch

import pyoracle as O
import workloads as W

pytestmark = pytest.mark.gpu

FORMATS = ["CSRScalar", "CSRAdaptive", "Ellpack", "SlicedEllpack", "ChunkedEllpack", "BiEllpack"]


def oracle_columns(rp, c, v, X):
    seg = O.Segments("CSR", np.diff(rp))
    ov, oc = seg.convert(rp, c, v)
    return np.stack([seg.spmv(ov, oc, np.ascontiguousarray(X[:, j])) for j in range(X.shape[1])], axis=1)


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("k", [1, 3, 16, 40])
def test_block_product_equals_oracle_per_column(tnl, dev, fmt, k):
    rp, c, v = W.irregular(3001, 9.0, 1.0, 300, seed=k)
    n = len(rp) - 1
    X = np.random.default_rng(k).uniform(-1, 1, (n, k))
    want = oracle_columns(rp, c, v, X)
    A = tnl.SparseMatrix.from_csr(rp, c, v, format=fmt, dtype="f64")
    Y = torch.full((n, k), np.nan, dtype=torch.float64, device=dev)
    A.vectorProductMulti(torch.tensor(X, device=dev), Y)
    torch.cuda.synchronize()
    assert np.array_equal(Y.cpu().numpy(), want), fmt


@pytest.mark.parametrize("fmt", ["CSRAdaptive", "SlicedEllpack"])
def test_block_product_keepers_and_row_range(tnl, dev, fmt):
    rp, c, v = W.laplacian_3d(14)
    n = len(rp) - 1
    k = 5
    rng = np.random.default_rng(3)
    X = rng.uniform(-1, 1, (n, k))
    Y0 = rng.uniform(-1, 1, (n, k))
    AX = oracle_columns(rp, c, v, X)
    A = tnl.SparseMatrix.from_csr(rp, c, v, format=fmt, dtype="f64")
    Xd = torch.tensor(X, device=dev)
    for alpha, beta in ((1.0, 0.0), (-2.0, 0.0), (1.0, 0.5), (0.25, -1.5)):
        Y = torch.tensor(Y0, device=dev)
        A.vectorProductMulti(Xd, Y, alpha, beta, 100, 2000)
        got = Y.cpu().numpy()
        want = Y0.copy()
        want[100:2000] = beta * Y0[100:2000] + alpha * AX[100:2000] if beta else alpha * AX[100:2000]
        np.testing.assert_allclose(got, want, rtol=1e-14, atol=1e-13)
        assert np.array_equal(got[:100], Y0[:100]) and np.array_equal(got[2000:], Y0[2000:])


@pytest.mark.parametrize("dt", ["f32", "bf16"])
def test_block_product_low_precision(tnl, dev, dt):
    rp, c, v = W.convection_diffusion_3d(16, 10.0)
    n = len(rp) - 1
    k = 8
    X = np.random.default_rng(5).uniform(-1, 1, (n, k)).astype(np.float32)
    A = tnl.SparseMatrix.from_csr(rp, c, v, format="ChunkedEllpack", dtype=dt)
    Y = torch.zeros((n, k), dtype=torch.float32, device=dev)
    A.vectorProductMulti(torch.tensor(X, device=dev), Y)
    y1 = torch.zeros(n, dtype=torch.float32, device=dev)
    got = Y.cpu().numpy()
    for j in range(k):
        # the one-vector product of the same matrix on column j: same order, same bits
        A.vectorProduct(torch.tensor(np.ascontiguousarray(X[:, j]), device=dev), y1)
        ref = y1.cpu().numpy()
        scale = np.abs(v).max() * 7
        assert np.max(np.abs(got[:, j] - ref)) <= 1e-6 * scale


def test_block_product_refusals(tnl, dev):
    rp, c, v = W.laplacian_3d(6)
    n = len(rp) - 1
    A = tnl.SparseMatrix.from_csr(rp, c, v, format="CSRScalar", dtype="f64")
    for k in (65, 100):
        with pytest.raises(tnl.TnlHipError):
            A.vectorProductMulti(torch.zeros((n, k), dtype=torch.float64, device=dev),
                                 torch.zeros((n, k), dtype=torch.float64, device=dev))
    rows = np.repeat(np.arange(n), np.diff(rp))
    keep = c <= rows
    lrp = np.concatenate([[0], np.cumsum(np.bincount(rows[keep], minlength=n))]).astype(np.int32)
    S = tnl.SparseMatrix.symmetric_from_csr(lrp, c[keep], v[keep], format="CSRScalar")
    with pytest.raises(tnl.TnlHipError):
        S.vectorProductMulti(torch.zeros((n, 2), dtype=torch.float64, device=dev),
                             torch.zeros((n, 2), dtype=torch.float64, device=dev))


@pytest.mark.parametrize("fmt", FORMATS)
def test_block_product_without_columns(tnl, dev, fmt):
    """A matrix with no columns (every row empty) and an empty X: only the keepers act, and X,
    which holds no entry, is never read."""
    n, k = 70, 5
    rp = np.zeros(n + 1, np.int32)
    A = tnl.SparseMatrix.from_csr(rp, np.zeros(0, np.int32), np.zeros(0), columns=0, format=fmt, dtype="f64")
    Y0 = np.random.default_rng(4).uniform(-1, 1, (n, k))
    X = torch.zeros((0, k), dtype=torch.float64, device=dev)
    for alpha, beta in ((1.0, 0.0), (2.0, 0.5)):
        Y = torch.tensor(Y0, device=dev)
        A.vectorProductMulti(X, Y, alpha, beta)
        assert np.array_equal(Y.cpu().numpy(), beta * Y0), (fmt, alpha, beta)
        y = torch.tensor(Y0[:, 0].copy(), device=dev)
        A.vectorProduct(torch.zeros(0, dtype=torch.float64, device=dev), y, alpha, beta)
        assert np.array_equal(y.cpu().numpy(), beta * Y0[:, 0]), (fmt, alpha, beta)


def test_binary_product_without_columns(tnl, dev):
    n = 45
    rp = np.zeros(n + 1, np.int32)
    B = tnl.SparseMatrix.from_csr(rp, np.zeros(0, np.int32), None, columns=0, format="SlicedEllpack", dtype="binary")
    y0 = torch.arange(n, dtype=torch.int32, device=dev)
    for alpha, beta in ((1, 0), (3, 2)):
        y = y0.clone()
        B.vectorProduct(torch.zeros(0, dtype=torch.int32, device=dev), y, alpha, beta)
        assert torch.equal(y, beta * y0)


def test_block_product_unaligned_blocks_take_the_scalar_lanes(tnl, dev):
    """X and Y starting 8 bytes past a 16-byte boundary (FP64, k even) take the one-column-per-lane
    kernel instead of the 16-byte lanes; both give the oracle's bits."""
    rp, c, v = W.irregular(2501, 8.0, 1.0, 120, seed=21)
    n, k = len(rp) - 1, 6
    X = np.random.default_rng(21).uniform(-1, 1, (n, k))
    want = oracle_columns(rp, c, v, X)
    A = tnl.SparseMatrix.from_csr(rp, c, v, format="SlicedEllpack", dtype="f64")
    Xbig = torch.zeros(n * k + 1, dtype=torch.float64, device=dev)
    Xbig[1:] = torch.tensor(X.ravel(), device=dev)
    Ybig = torch.full((n * k + 1,), np.nan, dtype=torch.float64, device=dev)
    Xu, Yu = Xbig[1:].view(n, k), Ybig[1:].view(n, k)
    assert Xu.data_ptr() % 16 == 8 and Yu.data_ptr() % 16 == 8
    A.vectorProductMulti(Xu, Yu)
    Ya = torch.full((n, k), np.nan, dtype=torch.float64, device=dev)
    A.vectorProductMulti(torch.tensor(X, device=dev), Ya)
    torch.cuda.synchronize()
    assert np.array_equal(Yu.cpu().numpy(), want)
    assert np.array_equal(Ya.cpu().numpy(), want)


@pytest.mark.parametrize("fmt", ["CSRScalar", "Ellpack", "SlicedEllpack", "ChunkedEllpack"])
@pytest.mark.parametrize("dt", ["f64", "f32"])
@pytest.mark.parametrize("k", [3, 5, 7, 9, 12, 16, 17, 33, 64])
def test_short_rows_equal_the_columns_one_by_one(tnl, dev, fmt, dt, k):
    # 65 x 67 x 61 rows: ragged tiles, a walk of 8 tiles per wave in FP64 at k >= 33 and of 2 else, a few rows beyond
    # 8 slots (which keep the other kernel) in the CSR forms; X and Y at odd element offsets, so that 16-byte lanes
    # never divide a row; a row range that starts inside a tile; CSRScalar's one-vector product sums every row
    # in the same order with the same rounding
    rng = np.random.default_rng(k)
    for box, longs in (((65, 67, 61), fmt == "CSRScalar"), ((9, 5, 3), True)):
        rp, c, v = W._stencil(box[::-1], [(d, 1.0) for d in ((-1, 0, 0), (0, -1, 0), (0, 0, -1), (0, 0, 0), (0, 0, 1),
                                                            (0, 1, 0), (1, 0, 0))])
        n = len(rp) - 1
        rows = np.repeat(np.arange(n), np.diff(rp))
        key = rows.astype(np.int64) * n + c
        if longs:
            extra = rng.choice(n, 5, replace=False)
            key = np.unique(np.concatenate([key] + [r * n + rng.choice(n, 40) for r in extra.astype(np.int64)]))
        rows, c = key // n, (key % n).astype(np.int32)
        rp = np.zeros(n + 1, np.int32)
        np.cumsum(np.bincount(rows, minlength=n), out=rp[1:])
        v = rng.uniform(-1, 1, len(c))
        td = torch.float64 if dt == "f64" else torch.float32
        A = tnl.SparseMatrix.from_csr(rp, c, v, format=fmt, dtype=dt)
        B = tnl.SparseMatrix.from_csr(rp, c, v, format="CSRScalar", dtype=dt)
        X = torch.tensor(rng.uniform(-1, 1, n * k + 1), dtype=td, device=dev)[1:].view(n, k)
        Y0 = torch.tensor(rng.uniform(-1, 1, n * k + 1), dtype=td, device=dev)[1:].view(n, k)
        want = torch.stack([B.vectorProduct(X[:, j].contiguous(), torch.zeros(n, dtype=td, device=dev))
                            for j in range(k)], 1)
        Y = Y0.clone()
        A.vectorProductMulti(X, Y)
        assert torch.equal(Y, want), (box, "y = A x")
        for alpha, beta, lo, hi in ((-1.0, 1.0, 0, n), (0.5, -2.0, 7, n - 3)):
            Y = torch.empty(n * k + 1, dtype=td, device=dev)[1:].view(n, k).copy_(Y0)
            A.vectorProductMulti(X, Y, alpha, beta, lo, hi)
            ref = Y0.double() * beta + alpha * want.double()
            eps = 2.0 ** (-50 if dt == "f64" else -21)
            assert (Y[lo:hi].double() - ref[lo:hi]).abs().max() <= eps * 8
            assert torch.equal(Y[:lo], Y0[:lo]) and torch.equal(Y[hi:], Y0[hi:])


def test_a_long_row_among_short_ones_costs_odd_widths_no_more(tnl, dev):
    """The walk for short rows (odd k) is not taken where a row holds more than 8 slots: k = 7 costs what k = 8 does in
    the other kernel (which takes it at this size), give or take; in the walk the long row alone cost 3.6 times that."""
    n, m = 300000, 20000
    i = np.arange(n)
    e = np.sort(np.random.default_rng(1).choice(np.arange(2, n), m, replace=False))
    cols = [np.concatenate([[0, 1], e]), *np.stack([i[:-2], i[1:-1], i[2:]], 1), np.array([n - 2, n - 1])]
    rp = np.zeros(n + 1, np.int32)
    np.cumsum([len(c) for c in cols], out=rp[1:])
    c = np.concatenate(cols).astype(np.int32)
    v = np.random.default_rng(2).uniform(-1, 1, len(c))
    A = tnl.SparseMatrix.from_csr(rp, c, v, format="CSRScalar", dtype="f64")
    took = {}
    for k in (7, 8):
        X = torch.tensor(np.random.default_rng(k).uniform(-1, 1, (n, k)), device=dev)
        Y = torch.zeros_like(X)
        for r in range(4):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            A.vectorProductMulti(X, Y)
            e1.record()
            e1.synchronize()
            took[k] = min(took.get(k, 1e9), e0.elapsed_time(e1))
        want = torch.zeros(n, dtype=torch.float64, device=dev)
        A.vectorProduct(X[:, k - 1].contiguous(), want)
        assert torch.equal(Y[:, k - 1], want)
    assert took[7] < 2 * took[8], took


@pytest.mark.parametrize("fmt,dt,k,box,aligned,longs", [
    ("SlicedEllpack", "f64", 16, (101, 100, 83), True, 0),   # 16-byte lanes, 8 tiles per wave from 100000 tiles on
    ("SlicedEllpack", "f64", 16, (100, 99, 79), True, 0),    # the same below that: the other kernel
    ("SlicedEllpack", "f64", 3, (1001, 1003, 1), False, 0),  # two lanes a row, four slots a loader
    ("Ellpack", "f64", 3, (1001, 1003, 1), False, 0),
    ("SlicedEllpack", "f32", 33, (65, 67, 93), False, 0),    # 8 tiles per wave in FP32
    ("CSRScalar", "f64", 7, (65, 67, 61), False, 0),
    ("CSRScalar", "f32", 5, (65, 67, 61), True, 0),
    ("SlicedEllpack", "f64", 7, (65, 67, 61), False, 3),     # rows beyond 8 slots: the other kernel
    ("Ellpack", "f32", 9, (65, 67, 61), False, 3),
])
def test_each_rule_of_the_short_row_walk(tnl, dev, fmt, dt, k, box, aligned, longs):
    """Every column equals the one-vector product of the same rows bit for bit, whole and over a ragged range."""
    d = [(-1, 0, 0), (0, -1, 0), (0, 0, -1), (0, 0, 0), (0, 0, 1), (0, 1, 0), (1, 0, 0)]
    rp, c, v = W._stencil(box, [(q, 1.0) for q in d if box[2] > 1 or q[2] == 0])
    n = len(rp) - 1
    rng = np.random.default_rng(k)
    if longs:
        at = rng.choice(n, longs, replace=False)
        key = np.repeat(np.arange(n, dtype=np.int64), np.diff(rp)) * n + c
        key = np.unique(np.concatenate([key] + [r * n + rng.choice(n, 13) for r in at.astype(np.int64)]))
        c = (key % n).astype(np.int32)
        np.cumsum(np.bincount(key // n, minlength=n), out=rp[1:])
    v = rng.uniform(-1, 1, len(c))
    td = torch.float64 if dt == "f64" else torch.float32
    A = tnl.SparseMatrix.from_csr(rp, c, v, format=fmt, dtype=dt)
    B = tnl.SparseMatrix.from_csr(rp, c, v, format="CSRScalar", dtype=dt)
    off = 0 if aligned else 1
    X = torch.rand(n * k + off, dtype=td, device=dev, generator=torch.Generator(dev).manual_seed(k))[off:].view(n, k)
    Y = torch.full((n * k + off,), float("nan"), dtype=td, device=dev)[off:].view(n, k)
    A.vectorProductMulti(X, Y)
    lo, hi = 5, n - 6
    Z = torch.full((n * k + off,), 2.0, dtype=td, device=dev)[off:].view(n, k)
    A.vectorProductMulti(X, Z, 1.0, 0.0, lo, hi)
    y = torch.zeros(n, dtype=td, device=dev)
    for j in range(k):
        B.vectorProduct(X[:, j].contiguous(), y)
        assert torch.equal(Y[:, j], y), j
        assert torch.equal(Z[lo:hi, j], y[lo:hi]), j
    assert (Z[:lo] == 2).all() and (Z[hi:] == 2).all()
