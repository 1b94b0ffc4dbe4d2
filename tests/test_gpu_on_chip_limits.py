"""Which solves run on chip: up to the sizes where that is the faster way."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CU_ROWS = 256 * 512  # one row per thread of 256 workgroups


def _tridiag(n):
    i = np.arange(n)
    row = np.concatenate([i[1:], i, i[:-1]])
    col = np.concatenate([i[:-1], i, i[1:]])
    val = np.concatenate([np.full(n - 1, -1.1), np.full(n, 3.0), np.full(n - 1, -0.9)])
    return _csr(n, row, col, val)


def _csr(n, row, col, val):
    o = np.lexsort((col, row))
    ptr = np.zeros(n + 1, np.int32)
    ptr[1:] = np.cumsum(np.bincount(row, minlength=n))
    return ptr, col[o].astype(np.int32), val[o]


def _runs_on_chip(ctx, A, b, outer, inner, **kw):
    from solver_cpp_amd import api
    before = ctx.on_chip()
    x, r, _ = api.solve(ctx, A, b, outer, inner, history=False, outer_eps=1e-10, outer_maxloop=300, **kw)
    assert r["status"] == 0 and r["relres_true"] < 1e-9
    after = ctx.on_chip()
    assert after["repeated"] == before["repeated"]
    return after["solves"] > before["solves"]


@pytest.mark.parametrize("prec", [64, 32])
@pytest.mark.parametrize("n", [2 * CU_ROWS, 2 * CU_ROWS + 1, 4 * CU_ROWS])
def test_bicg_takes_two_rows_per_thread(ctx, n, prec):
    from solver_cpp_amd import api
    A = api.Matrix(ctx, *_tridiag(n), fp32=True, transpose=True)
    b = np.random.default_rng(71).uniform(-1, 1, n)
    got = _runs_on_chip(ctx, A, b, "vpgmres", "bicg", outer_restart=20, inner_maxloop=10, inner_precision=prec)
    assert got == (n <= 2 * CU_ROWS)
    A.close()


def _random_rows(n, pairs):
    # the diagonal, and both directions of `pairs` random permutations
    rng = np.random.default_rng(72)
    i = np.arange(n)
    row, col, val = [i], [i], [np.full(n, 2.2 * pairs)]
    for _ in range(pairs):
        p = rng.permutation(n)
        row, col, val = row + [i, p], col + [p, i], val + [np.full(n, -1.0)] * 2
    return _csr(n, np.concatenate(row), np.concatenate(col), np.concatenate(val))


def _box(nx, ny, nz):
    from solver_cpp_amd import gen
    ptr, col, val = gen.stencil(3, nx, ny, nz)
    return ptr, col, np.where(col == np.repeat(np.arange(nx * ny * nz), np.diff(ptr)), val + 1.0, val)


@pytest.mark.parametrize("outer,inner,kw", [("cg", "NO", {}),
                                            ("vpcg", "cg", dict(inner_maxloop=10, inner_precision=32))])
@pytest.mark.parametrize("name,make,yes", [
    ("random_7_two_rows", lambda: _random_rows(2 * CU_ROWS, 3), True),
    ("random_7_four_rows", lambda: _random_rows(2 * CU_ROWS + 1, 3), False),
    ("random_5_four_rows", lambda: _random_rows(4 * CU_ROWS, 2), False),
    ("random_3_four_rows", lambda: _random_rows(300_000, 1), True),
    ("thin_box", lambda: _box(2048, 16, 16), True),  # four neighbours in other workgroups, in runs
    ("cube", lambda: _box(70, 70, 70), True),
    ("line", lambda: _tridiag(4 * CU_ROWS), True),
    ("line_too_long", lambda: _tridiag(4 * CU_ROWS + 1), False),
])
def test_cg_with_four_rows_per_thread_gathers_runs(ctx, name, make, yes, outer, inner, kw):
    from solver_cpp_amd import api
    ptr, col, val = make()
    if name.startswith("line"):
        val = np.where(val < 0, -1.0, val)  # symmetric
    A = api.Matrix(ctx, ptr, col, val, fp32=True, spd=True)
    b = np.random.default_rng(73).uniform(-1, 1, len(ptr) - 1)
    assert _runs_on_chip(ctx, A, b, outer, inner, **kw) == yes
    A.close()


@pytest.mark.parametrize("outer,maxloop", [("cg", 300), ("cg", 2000), ("bicg", 300)])
def test_counted_bytes(ctx, outer, maxloop):
    # the matrix and the vectors once a launch of at most 1024 steps, and each
    # step's stores; by launches, the products and vector passes of every step
    from solver_cpp_amd import api
    n = 20_000
    ptr, col, val = _tridiag(n)
    nnz = len(col)
    A = api.Matrix(ctx, ptr, col, val, transpose=True)
    b = np.random.default_rng(74).uniform(-1, 1, n)
    x, r, _ = api.solve(ctx, A, b, outer, history=False, outer_eps=0.0, outer_maxloop=maxloop)
    launches = -(-r["steps"] // 1024)
    csr, sides = 12 * nnz + 4 * (n + 1), 1 if outer == "cg" else 2
    per_launch = sides * csr + (4 if outer == "cg" else 6) * 8 * n
    assert list(r["prof"]) == ["spmv64"] and r["spmv"] == sides * r["steps"]
    assert r["bytes"] == launches * per_launch + r["steps"] * 2 * sides * 8 * n
    A.close()
