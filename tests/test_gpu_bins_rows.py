"""Column blocks row by row: each row held to a bound of its own length, on A
and on A^T, in both precisions, before and after new values.

A row of m entries is within m eps times the sum of |a x| of the exact one (a
rounding of each product, m - 1 of the additions in any order), and so is the
FP64 sum it is compared with: 2 m eps is allowed, and an empty row is zero."""
import numpy as np
import pytest

from tests import _problems as P
from tests.test_gpu_bins import _matrix

pytestmark = pytest.mark.gpu

EPS = {64: 2.0 ** -53, 32: 2.0 ** -24}


def _two_sided():
    # heavy-tailed rows and columns: the matrix beside its own transpose
    import scipy.sparse as sp
    ptr, col, val = _matrix(8192, cap=7000)
    n = len(ptr) - 1
    S = sp.csr_matrix((val, col, ptr), shape=(n, n))
    C = sp.csr_matrix(S + sp.csr_matrix(S.T)[:, ::-1].tocsr())
    C.sort_indices()
    return C


def _products(A, C, trans, seed):
    M = C.T.tocsr() if trans else C
    n = C.shape[0]
    x = np.random.default_rng(seed).standard_normal(n)
    m = np.diff(M.indptr)
    for prec, dt in ((64, np.float64), (32, np.float32)):
        xp = x.astype(dt)
        v = M.data.astype(dt).astype(np.float64)
        ref = type(M)((v, M.indices, M.indptr), shape=M.shape) @ xp.astype(np.float64)
        y = A.spmv(xp, trans=trans, precision=prec).astype(np.float64)
        bound = 2 * m * EPS[prec] * P.row_abs_bound(M.indptr, M.indices, v, xp.astype(np.float64))
        assert np.all(np.abs(y - ref) <= bound * (1 + 1e-6) + 1e-37)
        assert not y[m == 0].any()


def test_every_row_of_both_sides(ctx):
    from solver_cpp_amd import api
    C = _two_sided()
    n, nnz = C.shape[0], C.nnz
    A = api.Matrix(ctx, C.indptr.astype(np.int32), C.indices.astype(np.int32), C.data, transpose=True, fp32=True)
    for trans in (False, True):
        for prec in (64, 32):
            sv = prec // 8
            assert A.spmv_bytes(trans, prec) == (3 * sv + 4) * nnz + 4 * (n + 1) + 2 * sv * n
        _products(A, C, trans, 31 + trans)
    C.data[:] = np.random.default_rng(33).standard_normal(nnz)
    A.update_values(C.data)
    for trans in (False, True):
        _products(A, C, trans, 34 + trans)
    A.close()
