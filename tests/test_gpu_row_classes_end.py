"""New values that end a matrix's row classes: up to 32 classes become row
patterns in place (classes of one list of offsets share a pattern), and every
product equals the int32 columns' bit for bit."""
import numpy as np
import pytest

from tests.test_gpu_row_classes import SEVEN, _box, _const, _csr

pytestmark = pytest.mark.gpu


def _cases():
    yield "one_class", [[(i, 2.0)] for i in range(5000)]
    yield "7_point", _box((13, 11, 17), SEVEN, _const)
    # 20 classes of three lists
    yield "materials", [[(i, 1.0 + i % 10)] if i % 3 == 0 else
                        [(i, 1.0 + i % 5), (i + 1, -1.0)] if i % 3 == 1 else
                        [(i - 1, -1.0), (i, 3.0 + i % 5)] for i in range(5100)]
    yield "32_lists", [[(i, 1.0), (i + i % 31 + 1, 0.5)] if i < 5000 else [(i, 1.0)] for i in range(5040)]
    yield "empty_rows", [[] if i % 3 == 0 else [(i, 2.0), (i - 1, -0.5)] for i in range(9000)]
    yield "8_entries", [[(i + k * 7 % 8, 1.0 + k) for k in range(8)] if i < 4000 else [(i, 1.0)]
                        for i in range(4100)]


@pytest.mark.parametrize("name,rows", list(_cases()), ids=[c[0] for c in _cases()])
def test_classes_become_patterns(ctx, name, rows):
    from solver_cpp_amd import api
    ptr, col, val = _csr(rows)
    n, nnz = len(rows), len(col)
    A = api.Matrix(ctx, ptr, col, val, transpose=True, fp32=True)
    B = api.Matrix(ctx, ptr, col, val, transpose=True, fp32=True, layout="col32")
    assert A.spmv_bytes() == 17 * n
    rng = np.random.default_rng(85)
    x, u = rng.standard_normal(n), rng.standard_normal(n)
    f = x.astype(np.float32)
    for k, v in enumerate((2.0 * val, rng.standard_normal(nnz), rng.standard_normal(nnz), val)):
        A.update_values(v)
        B.update_values(v)
        for trans in (False, True):
            assert np.array_equal(A.spmv(x, trans=trans), B.spmv(x, trans=trans))
            assert np.array_equal(A.spmv(f, trans=trans, precision=32), B.spmv(f, trans=trans, precision=32))
        for a, b in zip(A.kskip_basis(1, x, u), B.kskip_basis(1, x, u)):
            assert np.array_equal(a, b, equal_nan=True)
        # the classes agree in 2 val, then end for good
        assert A.spmv_bytes() == (17 * n if k == 0 else 18 * n + 8 * nnz)
    A.close()
    B.close()


def test_one_value_ends_both_sides(ctx):
    # values that repeat by rows, then a single one that differs in the middle
    from solver_cpp_amd import api
    n = 6000
    ptr, col, val = _csr([[(i, 2.0), ((i + 1) % n, 1.0)] for i in range(n)])
    A = api.Matrix(ctx, ptr, col, val, transpose=True)
    assert A.spmv_bytes() == A.spmv_bytes(True) == 17 * n
    for v, kept in ((np.tile([5.0, 7.0], n), True), (np.where(np.arange(2 * n) == n, 9.0, val), False)):
        A.update_values(v)
        for trans in (False, True):
            assert (A.spmv_bytes(trans) == 17 * n) == kept
        B = api.Matrix(ctx, ptr, col, v, transpose=True, layout="col32")
        x = np.random.default_rng(86).standard_normal(n)
        for trans in (False, True):
            assert np.array_equal(A.spmv(x, trans=trans), B.spmv(x, trans=trans))
        B.close()
    A.close()
