"""Products and solves that read int16 offsets and delta-coded columns.

Matrices with few lists of column offsets are read as row patterns or classes
instead, so each matrix here has a column whose offset takes fifty values, and
`spmv_bytes` is asserted to be the 16-bit format's.  Every result equals the
int32 columns' bit for bit (the same gathers in the same order), and products
the oracle's (rows of at most 8 entries)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _csr(n, row, col, val=None, seed=51):
    o = np.lexsort((col, row))
    ptr = np.zeros(n + 1, np.int32)
    ptr[1:] = np.cumsum(np.bincount(row, minlength=n))
    if val is None:
        val = np.random.default_rng(seed).standard_normal(len(col))
    return ptr, col[o].astype(np.int32), val[o]


def _band(n, offsets, extra):
    """Entries at row + d, d in offsets, and one at row + extra + (0 .. 49)."""
    i = np.arange(n)
    row = np.concatenate([i] * (len(offsets) + 1))
    col = np.concatenate([i + d for d in offsets] + [i + extra + i * 7 % 50])
    ok = (col >= 0) & (col < n)
    return _csr(n, row[ok], col[ok])


def _format(n, nnz, prec, ib):
    sv = prec // 8
    return (sv + ib) * nnz + 4 * (n + 1) + 2 * sv * n


def _check(ctx, oracle, ptr, col, val, ib, ibt, layout="auto"):
    from solver_cpp_amd import api
    n, nnz = len(ptr) - 1, len(col)
    A = api.Matrix(ctx, ptr, col, val, transpose=True, fp32=True, layout=layout)
    B = api.Matrix(ctx, ptr, col, val, transpose=True, fp32=True, layout="col32")
    x = np.random.default_rng(52).standard_normal(n)
    x32 = x.astype(np.float32)
    otp, otc, otv = oracle.transpose(ptr, col, val)
    short = np.diff(ptr).max() <= 8 and np.diff(otp).max() <= 8
    for trans, (p, c, v), b in ((False, (ptr, col, val), ib), (True, (otp, otc, otv), ibt)):
        for prec in (64, 32):
            assert A.spmv_bytes(trans, prec) == _format(n, nnz, prec, b) and A.index_bytes(trans, prec) == b
        y, y32 = A.spmv(x, trans=trans), A.spmv(x32, trans=trans, precision=32)
        assert np.array_equal(y, B.spmv(x, trans=trans))
        assert np.array_equal(y32, B.spmv(x32, trans=trans, precision=32))
        if short:
            assert np.array_equal(y, oracle.spmv(p, c, v, x))
            assert np.array_equal(y32, oracle.spmv_f32(p, c, v.astype(np.float32), x32))
    for a, b in zip(A.kskip_basis(1, x, x[::-1].copy()), B.kskip_basis(1, x, x[::-1].copy())):
        assert np.array_equal(a, b, equal_nan=True)
    A.close()
    B.close()


@pytest.mark.parametrize("layout", ["auto", "delta"])
@pytest.mark.parametrize("reach", [32767, 32768])
def test_int16_offsets_at_their_limit(ctx, oracle, reach, layout):
    # beyond +-32767: delta codes; six entries a row, and eight (more than are
    # gathered ahead of the next tile's loads in FP64)
    for more in ([], [-500, 400]):
        _check(ctx, oracle, *_band(70_000, [-reach, -3, 0, 1, reach] + more, 3), 2, 2, layout)


@pytest.mark.parametrize("offsets,extra,ib,ibt", [
    ([-49152, -3, 0, 1, 49152], 3, 2, 2),   # first column at row - 49152: the lowest code
    ([-49153, -3, 0, 1, 49153], 3, 4, 4),   # one below
    ([0, 65535], 65536, 2, 4),              # gap 65535 in A; A^T's first columns lie too far below
    ([0, 65536], 65537, 4, 4),              # gap 65536
    ([16383, 40000], 16385, 2, 2),          # first column at row + 16383: the highest code
    ([16384, 40000], 16386, 4, 2),          # one above in A; A^T's columns lie below the row
])
def test_delta_codes_at_their_limits(ctx, oracle, offsets, extra, ib, ibt):
    _check(ctx, oracle, *_band(140_000, offsets, extra), ib, ibt)


def test_unsorted_rows(ctx, oracle):
    # A's rows in descending order: int32 columns (far) or int16 offsets
    # (near); A^T, built sorted, has delta codes or int16 offsets
    for reach, ib in ((40000, 4), (30000, 2)):
        ptr, col, val = _band(100_000, [-reach, -1, 0, 1, reach], 3)
        for i in range(len(ptr) - 1):
            col[ptr[i]:ptr[i + 1]] = col[ptr[i]:ptr[i + 1]][::-1].copy()
        _check(ctx, oracle, ptr, col, val, ib, 2)


@pytest.mark.parametrize("layout", ["auto", "delta"])
def test_two_lanes_a_row(ctx, oracle, layout):
    # 18 entries a row: no delta codes, int16 offsets where they fit
    for reach, ib in ((40000, 4), (30000, 2)):
        _check(ctx, oracle, *_band(100_000, [-reach] + list(range(-8, 7)) + [reach], 8), ib, ib, layout)


def _system(n, symmetric):
    """Neighbours along a line and one edge a pair of rows of varying length, diagonally dominant."""
    rng = np.random.default_rng(53)
    k = np.arange(n // 2)
    a = np.concatenate([np.arange(n - 1), 2 * k])
    b = np.concatenate([np.arange(1, n), 2 * k + 3 + 2 * (k * 7 % 50)])
    a, b = a[b < n], b[b < n]
    w = -rng.uniform(0.5, 1.5, len(a))
    row, col = np.concatenate([a, b]), np.concatenate([b, a])
    val = np.concatenate([w, w if symmetric else 1.3 * w])
    diag = np.bincount(row, -val, n) * (1.0 if symmetric else 1.15) + 0.5
    row, col, val = np.concatenate([row, np.arange(n)]), np.concatenate([col, np.arange(n)]), np.concatenate([val, diag])
    return _csr(n, row, col, val)


@pytest.mark.parametrize("outer,inner,kw", [
    ("cg", "NO", {}), ("bicg", "NO", {}), ("gmres", "NO", dict(outer_restart=21)),
    ("kskipcg", "NO", dict(outer_kskip=2)),
    ("vpgmres", "gmres", dict(outer_restart=21, inner_maxloop=11, inner_restart=12, inner_precision=32)),
])
def test_solves_in_every_index_format(ctx, outer, inner, kw):
    # more rows than run on chip, and more tiles than workgroups are resident
    from solver_cpp_amd import api
    n = 600_000
    sym = outer in ("cg", "kskipcg")
    ptr, col, val = _system(n, sym)
    nnz = len(col)
    b = np.random.default_rng(54).uniform(-1, 1, n)
    out = []
    for layout, ib in (("auto", 2), ("delta", 2), ("col32", 4)):
        A = api.Matrix(ctx, ptr, col, val, fp32=True, spd=sym, transpose=not sym, layout=layout)
        for prec in (64, 32):
            assert A.spmv_bytes(False, prec) == _format(n, nnz, prec, ib)
            assert sym or A.spmv_bytes(True, prec) == _format(n, nnz, prec, ib)
        x, r, h = api.solve(ctx, A, b, outer, inner, outer_eps=1e-10, outer_maxloop=5000, **kw)
        assert r["status"] == 0 and r["relres_true"] < 1e-8
        out.append((x, h))
        A.close()
    for x, h in out[:2]:
        assert np.array_equal(x, out[2][0]) and np.array_equal(h, out[2][1])
