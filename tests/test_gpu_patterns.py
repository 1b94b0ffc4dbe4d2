"""The row-pattern column format (at most 32 distinct lists of column offsets
per matrix) against the int32 format, bit for bit, and where it applies."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _csr(rows, seed):
    ptr = np.zeros(len(rows) + 1, np.int32)
    ptr[1:] = np.cumsum([len(r) for r in rows])
    col = np.array([c for r in rows for c in r], np.int32)
    return ptr, col, np.random.default_rng(seed).standard_normal(len(col))


def _band(n, offsets):
    return [[i + d for d in offsets if 0 <= i + d < n] for i in range(n)]


def _cases():
    yield "one_row", [[0]], True
    yield "no_entries_but_one", [[], [1], [], []], True
    yield "unsorted_and_repeated", _band(1500, [3, 0, -2, 0, 3]), True
    # 27-point stencil, 3-D: two lanes per row, a ragged last tile
    off = [x + 9 * (y + 11 * z) for z in (-1, 0, 1) for y in (-1, 0, 1) for x in (-1, 0, 1)]
    yield "27_point", _band(9 * 11 * 13, off), True
    inner = [[i + d for d in off] if 200 <= i < 1000 else [i] for i in range(1287)]
    yield "27_point_inner", inner, True
    # m patterns of the diagonal and one entry 1 .. m - 1 away, and the last row's
    for m, ok in ((31, True), (32, False)):
        yield f"{m + 1}_patterns", [[i, (i + i % m + 1)] if i + m < 3000 else [i, i + 1] if i < 2999 else [i, i - 1]
                                    for i in range(3000)], ok
    # table limit: 1 + 32 + P * 256 <= 1024 ints
    for p, ok in ((3, True), (4, False)):
        yield f"{p}_of_256", [list(range(256))] + [[i] + [i + 1] * (i % 3 > 0) + [i - 1] * (i % 3 > 4 - p + 1)
                                                   for i in range(1, 2999)] + [[2999]], ok
    yield "tile_of_2041", [[i + k for k in range(13)] if i < 157 * 40 else [i] for i in range(157 * 40 + 300)], True


@pytest.mark.parametrize("name,rows,applies", list(_cases()), ids=[c[0] for c in _cases()])
def test_row_patterns_same_as_int32(ctx, oracle, name, rows, applies):
    from solver_cpp_amd import api
    ptr, col, val = _csr(rows, 71)
    n, nnz = len(rows), len(col)
    A = api.Matrix(ctx, ptr, col, val, transpose=True, fp32=True, layout="auto")
    B = api.Matrix(ctx, ptr, col, val, transpose=True, fp32=True, layout="col32")
    assert (A.spmv_bytes() == 8 * nnz + 2 * n + 16 * n) == (applies and A.info()["spmv_kind"] == 0)
    rng = np.random.default_rng(72)
    x = rng.standard_normal(n)
    for trans in (False, True):
        assert np.array_equal(A.spmv(x, trans=trans), B.spmv(x, trans=trans))
        x32 = x.astype(np.float32)
        assert np.array_equal(A.spmv(x32, trans=trans, precision=32), B.spmv(x32, trans=trans, precision=32))
    if max(len(r) for r in rows) <= 8:
        assert np.array_equal(A.spmv(x), oracle.spmv(ptr, col, val, x))
    # the two-input product and the refresh of the values
    p = rng.standard_normal(n)
    for a, b in zip(A.kskip_basis(1, x, p), B.kskip_basis(1, x, p)):
        assert np.array_equal(a, b, equal_nan=True)
    v2 = rng.standard_normal(nnz)
    A.update_values(v2)
    B.update_values(v2)
    assert np.array_equal(A.spmv(x), B.spmv(x)) and np.array_equal(A.spmv(x, trans=True), B.spmv(x, trans=True))
    A.close()
    B.close()


def test_row_patterns_off_for_the_other_layouts(ctx):
    # an explicit delta or int32 format, and the other kernels, keep their own indices
    from solver_cpp_amd import api
    ptr, col, val = _csr(_band(4000, [-1, 0, 1]), 73)
    n, nnz = 4000, len(col)
    for layout, ib in (("delta", 2), ("col32", 4), ("wave", 4), ("vector", 4), ("merge", 4)):
        A = api.Matrix(ctx, ptr, col, val, layout=layout)
        assert A.spmv_bytes() == (8 + ib) * nnz + 4 * (n + 1) + 16 * n
        A.close()
