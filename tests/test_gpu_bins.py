"""Column blocks (two-pass products with matrices whose rows gather x from all
over) against the merge path and plain FP64 sums, over row lengths at the edges
of its ways to sum a row, segments and column blocks.

A row of m terms differs from the FP64 sum by at most m eps sum |a x| in each
order of its additions, and one rounding of the products: 4 m eps is allowed,
as for the other layouts; the SDDMM is one product per entry, exact either
way."""
import numpy as np
import pytest

from tests import _problems as P

pytestmark = pytest.mark.gpu

EPS64, EPS32 = 2.0 ** -53, 2.0 ** -24


def _matrix(longest, cap=1 << 20):
    # 24 entries per row, and rows of every length at which the summation
    # changes; columns anywhere, but none in the third block of 16384; the
    # last block is a partial one, the last row empty
    n = 393216 + 5000
    rng = np.random.default_rng(17)
    cnt = np.full(n, 27)
    special = [0, 1, 2, 15, 16, 17, 63, 64, 65, 255, 256, 257, 1000, 8191, longest, 0, 8000, 300, 5]
    cnt[:len(special)] = special
    cnt[200000:200000 + len(special)] = special[::-1]
    cnt[300000:310000] = 0
    cnt[310000:312000] = rng.integers(0, 300, 2000)
    cnt[-1] = 0
    cnt = np.minimum(cnt, cap)
    ptr = np.zeros(n + 1, np.int32)
    ptr[1:] = np.cumsum(cnt)
    col = rng.integers(0, n - 16384, ptr[-1])
    col = (col + 16384 * (col >= 32768)).astype(np.int32)
    return ptr, col, rng.standard_normal(ptr[-1])


def _check(ctx, ptr, col, val, kind):
    import scipy.sparse as sp
    from solver_cpp_amd import api
    n, nnz = len(ptr) - 1, len(col)
    A = api.Matrix(ctx, ptr, col, val, transpose=True, fp32=True)
    assert A.info()["spmv_kind"] == kind
    rng = np.random.default_rng(18)
    x, u = rng.standard_normal(n), rng.standard_normal(n)
    m = int(np.diff(ptr).max())
    S = sp.csr_matrix((val, col, ptr), shape=(n, n))
    bound = P.row_abs_bound(ptr, col, val, x)
    y = A.spmv(x)
    assert np.all(np.abs(y - S @ x) <= 4 * m * EPS64 * bound + 1e-300)
    assert np.array_equal(y, A.spmv(x))
    x32, v32 = x.astype(np.float32), val.astype(np.float32)
    y32 = A.spmv(x32, precision=32)
    S32 = sp.csr_matrix((v32.astype(np.float64), col, ptr), shape=(n, n))
    assert np.all(np.abs(y32.astype(np.float64) - S32 @ x32.astype(np.float64)) <= 4 * m * EPS32 * bound + 1e-30)
    rows = np.repeat(np.arange(n), np.diff(ptr))
    assert np.array_equal(A.sddmm(-0.75, u, x), -0.75 * u[rows] * x[col])
    # the two-input product and new values
    Ar, Ap = A.kskip_basis(1, x, u)
    assert np.array_equal(Ar[0], y) and np.array_equal(Ap[0], A.spmv(u))
    w = rng.standard_normal(nnz)
    A.update_values(w)
    S = sp.csr_matrix((w, col, ptr), shape=(n, n))
    assert np.all(np.abs(A.spmv(x) - S @ x) <= 4 * m * EPS64 * P.row_abs_bound(ptr, col, w, x) + 1e-300)
    y32 = A.spmv(x32, precision=32)
    S32 = sp.csr_matrix((w.astype(np.float32).astype(np.float64), col, ptr), shape=(n, n))
    bound = P.row_abs_bound(ptr, col, w, x)
    assert np.all(np.abs(y32.astype(np.float64) - S32 @ x32.astype(np.float64)) <= 4 * m * EPS32 * bound + 1e-30)
    A.close()


@pytest.mark.parametrize("longest,kind", [(8192, 3), (8193, 2)])
def test_products(ctx, longest, kind):
    # a row longer than a segment keeps the merge path
    _check(ctx, *_matrix(longest), kind)


def test_both_sides(ctx):
    # A and A^T in column blocks: the matrix above beside its own transpose
    import scipy.sparse as sp
    from solver_cpp_amd import api
    ptr, col, val = _matrix(8192, cap=7000)
    n = len(ptr) - 1
    S = sp.csr_matrix((val, col, ptr), shape=(n, n))
    B = sp.csr_matrix(S.T)[:, ::-1].tocsr()
    C = sp.csr_matrix(S + B)
    C.sort_indices()
    A = api.Matrix(ctx, C.indptr.astype(np.int32), C.indices.astype(np.int32), C.data, transpose=True)
    x = np.random.default_rng(19).standard_normal(n)
    Ct = C.T.tocsr()
    m, mt = int(np.diff(C.indptr).max()), int(np.diff(Ct.indptr).max())
    assert np.all(np.abs(A.spmv(x) - C @ x) <= 4 * m * EPS64 * (abs(C) @ np.abs(x)) + 1e-300)
    assert np.all(np.abs(A.spmv(x, trans=True) - Ct @ x) <= 4 * mt * EPS64 * (abs(Ct) @ np.abs(x)) + 1e-300)
    A.close()


@pytest.mark.parametrize("outer,inner,kw", [
    ("gmres", "NO", dict(outer_restart=11)), ("bicg", "NO", {}),
    ("vpgmres", "gmres", dict(outer_restart=11, inner_maxloop=6, inner_restart=7, inner_precision=32)),
])
def test_solves(ctx, outer, inner, kw):
    # every epilogue a solver puts on the product: the same solution as on the
    # merge path (diagonally dominant: a handful of steps)
    import scipy.sparse as sp
    from solver_cpp_amd import api
    ptr, col, val = _matrix(8192, cap=7000)
    n = len(ptr) - 1
    S = sp.csr_matrix((val, col, ptr), shape=(n, n))
    d = np.asarray(abs(S).sum(axis=1)).ravel() + np.asarray(abs(S).sum(axis=0)).ravel() + 1.0
    D = sp.diags(1.0 / d)
    T = sp.csr_matrix(D @ S * 0.9 + sp.identity(n))
    T.sort_indices()
    p, c, v = T.indptr.astype(np.int32), T.indices.astype(np.int32), T.data
    b = np.random.default_rng(20).uniform(-1, 1, n)
    out = []
    for layout in ("auto", "merge"):
        A = api.Matrix(ctx, p, c, v, transpose=True, fp32=True, layout=layout)
        assert A.info()["spmv_kind"] == (3 if layout == "auto" else 2)
        out.append(api.solve(ctx, A, b, outer, inner, outer_eps=1e-12, outer_maxloop=200, **kw))
        A.close()
    (x, r, h), (y, s, g) = out
    assert r["status"] == s["status"] == 0 and abs(r["iters"] - s["iters"]) <= 1
    assert np.linalg.norm(x - y) <= 1e-10 * np.linalg.norm(y)


@pytest.mark.parametrize("where", ["first", "middle", "last"])
def test_segments_without_entries(ctx, where):
    # two whole segments (4096 rows) of empty rows: they have no column block's run
    n = 393216 + 5000
    cnt = np.full(n, 28)
    cnt[50000:52000] = np.random.default_rng(19).integers(0, 300, 2000)
    cnt[60000] = 8000
    at = dict(first=0, middle=200000, last=n - 9000)[where]
    cnt[at:at + 9000] = 0
    ptr = np.zeros(n + 1, np.int32)
    ptr[1:] = np.cumsum(cnt)
    rng = np.random.default_rng(20)
    _check(ctx, ptr, rng.integers(0, n, ptr[-1]).astype(np.int32), rng.standard_normal(ptr[-1]), 3)
