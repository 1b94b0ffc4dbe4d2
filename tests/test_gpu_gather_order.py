"""Products whose gathers go out behind the next tile's loads (short rows, and
rows that gather from all over) as well as ahead of it, in every index format,
against the oracle: rows of at most 8 entries bit for bit, longer ones within the
row-sum bound (a row of m terms: 4 m eps of the sum of |a x|)."""
import numpy as np
import pytest

from tests import _problems as P

pytestmark = pytest.mark.gpu

EPS64, EPS32 = 2.0 ** -53, 2.0 ** -24


def _csr(rows):
    ptr = np.zeros(len(rows) + 1, np.int32)
    ptr[1:] = np.cumsum([len(r) for r in rows])
    col = np.concatenate([np.asarray(r, np.int64) for r in rows]).astype(np.int32)
    return ptr, col, np.random.default_rng(91).standard_normal(len(col))


def _band(n, offsets, extra=0):
    return [[i + d for d in offsets if 0 <= i + d < n] + ([i + max(offsets) + 1 + i * 7 % extra]
            if extra and i + max(offsets) + 1 + i * 7 % extra < n else []) for i in range(n)]


def _random(n, lo, hi, reach=None, seed=92):
    rng = np.random.default_rng(seed)
    out = []
    for i in range(n):
        m = rng.integers(lo, hi + 1)
        a, b = (0, n) if reach is None else (max(0, i - reach), min(n, i + reach + 1))
        out.append(np.sort(rng.choice(b - a, min(m, b - a), replace=False)) + a)
    return out


def _dense_blocks(n, k):
    return [list(range(i // k * k, min(n, i // k * k + k))) for i in range(n)]


CASES = {
    "diagonal": lambda: _band(5000, [0]),
    "two_diagonals": lambda: _band(5000, [0, 3]),
    "three_diagonals": lambda: _band(5000, [-1, 0, 1]),
    "two_columns_one_varying": lambda: _band(5000, [0], 60),
    "three_columns_one_varying": lambda: _band(5000, [0, 1], 60),
    "four_columns_one_varying": lambda: _band(5000, [-1, 0, 1], 60),
    "six_columns_one_varying": lambda: _band(5000, [-70, -1, 0, 1, 70], 60),
    "far_diagonals_one_varying": lambda: _band(80_000, [-39_000, 0, 39_000], 60),
    "random_1_to_3": lambda: _random(9000, 1, 3),
    "random_0_to_8": lambda: _random(9000, 0, 8),
    "random_1_to_19": lambda: _random(9000, 1, 19),
    "near_1_to_59": lambda: _random(4000, 1, 59, 500),
    "near_1_to_199": lambda: _random(1500, 1, 199, 400),
    "blocks_of_16": lambda: _dense_blocks(3000, 16),
    "blocks_of_40": lambda: _dense_blocks(3000, 40),
    "one_row_of_3000": lambda: [list(range(3000))] + _band(3000, [0, 1])[1:],
}


@pytest.mark.parametrize("layout", ["auto", "delta", "col32"])
@pytest.mark.parametrize("name", list(CASES))
def test_products(ctx, oracle, name, layout):
    from solver_cpp_amd import api
    ptr, col, val = _csr(CASES[name]())
    n = len(ptr) - 1
    A = api.Matrix(ctx, ptr, col, val, transpose=True, fp32=True, layout=layout)
    rng = np.random.default_rng(93)
    x, u = rng.standard_normal(n), rng.standard_normal(n)
    x32 = x.astype(np.float32)

    def check(val):
        tp, tc, tv = oracle.transpose(ptr, col, val)
        for trans, (p, c, v) in ((False, (ptr, col, val)), (True, (tp, tc, tv))):
            m = np.diff(p).max()
            y, y32 = A.spmv(x, trans=trans), A.spmv(x32, trans=trans, precision=32)
            o, o32 = oracle.spmv(p, c, v, x), oracle.spmv_f32(p, c, v.astype(np.float32), x32)
            if m <= 8:
                assert np.array_equal(y, o) and np.array_equal(y32, o32)
            else:
                bound = P.row_abs_bound(p, c, v, x)
                assert np.all(np.abs(y - o) <= 4 * m * EPS64 * bound + 1e-300)
                assert np.all(np.abs(y32.astype(np.float64) - o32) <= 4 * m * EPS32 * bound + 1e-30)
        Ar, Ap = A.kskip_basis(1, x, u)  # the two-input product
        assert np.array_equal(Ar[0], A.spmv(x)) and np.array_equal(Ap[0], A.spmv(u))
    check(val)
    w = rng.standard_normal(len(val))
    A.update_values(w)
    check(w)
    A.close()


@pytest.mark.parametrize("outer,inner,kw", [
    ("gmres", "NO", dict(outer_restart=11)), ("bicg", "NO", {}), ("gcr", "NO", dict(outer_restart=8)),
    ("vpgmres", "gmres", dict(outer_restart=11, inner_maxloop=8, inner_restart=9, inner_precision=32)),
])
@pytest.mark.parametrize("name", ["two_columns_one_varying", "random_1_to_19", "near_1_to_59"])
def test_solves_in_every_format(ctx, name, outer, inner, kw):
    # the fused products (dot, residual, projection): the same bits by 16-bit
    # and by int32 columns, and the true residual
    from solver_cpp_amd import api
    ptr, col, val = _csr(CASES[name]())
    n = len(ptr) - 1
    row = np.repeat(np.arange(n), np.diff(ptr))
    scale = np.bincount(row, np.abs(val), n) + np.bincount(col, np.abs(val), n) + 1.0
    import scipy.sparse as sp
    M = sp.csr_matrix((val / scale[row], col, ptr), shape=(n, n)) * 0.9 + sp.identity(n)
    M = sp.csr_matrix(M)
    M.sort_indices()
    b = np.random.default_rng(94).uniform(-1, 1, n)
    out = []
    ctx.set_wait_limit(0)  # by launches also where the system would fit on chip
    try:
        for layout in ("auto", "col32"):
            A = api.Matrix(ctx, M.indptr.astype(np.int32), M.indices.astype(np.int32), M.data, transpose=True,
                           fp32=True, layout=layout)
            x, r, h = api.solve(ctx, A, b, outer, inner, outer_eps=1e-11, outer_maxloop=400, **kw)
            assert r["status"] == 0
            assert np.linalg.norm(b - M @ x) <= 1e-10 * np.linalg.norm(b)
            out.append((x, h))
            A.close()
    finally:
        ctx.set_wait_limit(1 << 21)
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
