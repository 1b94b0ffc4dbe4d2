"""Products by row classes (a matrix whose rows repeat at most 128 lists of
offsets and values is read as one byte per row and a table) against the int32
format, bit for bit: where the format applies, what new values do to it, and
the solvers' fused products."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _csr(rows):
    """rows: lists of (column, value)"""
    ptr = np.zeros(len(rows) + 1, np.int32)
    ptr[1:] = np.cumsum([len(r) for r in rows])
    flat = [e for r in rows for e in r]
    return ptr, np.array([c for c, _ in flat], np.int32), np.array([v for _, v in flat], np.float64)


def _box(e, off, value):
    """Stencil on a box of edges e: neighbours off inside the box, value(offset, point)."""
    pts = [(x, y, z) for z in range(e[2]) for y in range(e[1]) for x in range(e[0])]
    rows = []
    for x, y, z in pts:
        r = []
        for d in off:
            q = (x + d[0], y + d[1], z + d[2])
            if all(0 <= a < b for a, b in zip(q, e)):
                r.append((q[0] + e[0] * (q[1] + e[1] * q[2]), value(d, (x, y, z))))
        rows.append(r)
    return rows


SEVEN = [(0, 0, -1), (0, -1, 0), (-1, 0, 0), (0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1)]


def _const(d, _):
    return 6.5 + 0.1 * sum(d) if d == (0, 0, 0) else -1.0 - 0.01 * d[0] - 0.3 * d[1] + 0.7 * d[2]


def _cases():
    yield "7_point", _box((13, 11, 17), SEVEN, _const), True
    yield "two_materials", _box((16, 16, 9), SEVEN, lambda d, q: _const(d, q) * (1 + 9 * (q[2] > 4))), True
    yield "varying", _box((13, 11, 17), SEVEN, lambda d, q: _const(d, q) * (1 + 1e-16 * 4 * (q[0] * q[1] * q[2]))), False
    yield "two_alternating", [[(i, 2.0 + i % 2), ((i + 1) % 6000, 0.5 - i % 2)] for i in range(6000)], True  # no parent
    for m, ok in ((128, True), (129, False)):
        yield f"{m}_classes", [[(i, 1.0 + i % m)] for i in range(5000)], ok
    for m, ok in ((8, True), (9, False)):  # entries of the longest row, unsorted
        yield f"{m}_entries", [[(i + k * 7 % m, 1.0 + k) for k in range(m)] if i % 5 and i < 4000 else [(i, 1.0)]
                               for i in range(4100)], ok
    yield "few_entries", [[(i, 2.0)] for i in range(4095)], False
    yield "enough_entries", [[(i, 2.0)] for i in range(4096)], True
    yield "empty_rows", [[] if i % 3 == 0 else [(i, 2.0), (i - 1, -0.5)] for i in range(9000)], True
    yield "signed_zero_inf_nan", [[(i, (0.0, -0.0, np.inf, np.nan)[i % 4])] for i in range(5000)], True


@pytest.mark.parametrize("name,rows,applies", list(_cases()), ids=[c[0] for c in _cases()])
def test_row_classes_same_as_int32(ctx, name, rows, applies):
    from solver_cpp_amd import api
    ptr, col, val = _csr(rows)
    n, nnz = len(rows), len(col)
    A = api.Matrix(ctx, ptr, col, val, transpose=True, fp32=True)
    B = api.Matrix(ctx, ptr, col, val, transpose=True, fp32=True, layout="col32")
    assert (A.spmv_bytes() == 17 * n) == (applies and A.info()["spmv_kind"] == 0)
    rng = np.random.default_rng(82)
    x, p = rng.standard_normal(n), rng.standard_normal(n)

    def same():
        for trans in (False, True):
            assert np.array_equal(A.spmv(x, trans=trans), B.spmv(x, trans=trans), equal_nan=True)
            f = x.astype(np.float32)
            assert np.array_equal(A.spmv(f, trans=trans, precision=32), B.spmv(f, trans=trans, precision=32),
                                  equal_nan=True)
        for a, b in zip(A.kskip_basis(1, x, p), B.kskip_basis(1, x, p)):
            assert np.array_equal(a, b, equal_nan=True)
    same()
    # new values: the same classes scaled, then every entry its own
    bytes_now = A.spmv_bytes()
    for k, v2 in enumerate((-1.5 * val, rng.standard_normal(nnz), val)):
        A.update_values(v2)
        B.update_values(v2)
        same()
        if k == 0:
            assert A.spmv_bytes() == bytes_now
        else:
            assert A.spmv_bytes() > 17 * n
    A.close()
    B.close()


@pytest.mark.parametrize("outer,inner,kw", [("gmres", "NO", dict(outer_restart=13)),
                                            ("bicg", "NO", {}), ("kskipcg", "NO", dict(outer_kskip=2)),
                                            ("vpgmres", "gmres", dict(outer_restart=9, inner_maxloop=8,
                                                                      inner_restart=9, inner_precision=32))])
def test_solves_same_as_int32(ctx, outer, inner, kw):
    # the fused products: dot, projection and deferred norm, two inputs
    from solver_cpp_amd import api
    ptr, col, val = _csr(_box((40, 37, 29), SEVEN, lambda d, q: 6.0 if d == (0, 0, 0) else -1.0 + 0.2 * (
        outer in ("gmres", "bicg")) * d[0]))
    b = np.random.default_rng(83).uniform(-1, 1, len(ptr) - 1)
    out = []
    for layout in ("auto", "col32"):
        A = api.Matrix(ctx, ptr, col, val, transpose=True, fp32=True, spd=outer == "kskipcg", layout=layout)
        x, r, h = api.solve(ctx, A, b, outer, inner, outer_eps=1e-9, outer_maxloop=2000, **kw)
        assert r["status"] == 0
        out.append((x, h))
        A.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


def test_borrowed_values_are_read_in_place(ctx):
    import torch
    from solver_cpp_amd import api
    ptr, col, val = (torch.from_numpy(a).cuda() for a in _csr(_box((13, 11, 17), SEVEN, _const)))
    A = api.Matrix(ctx, ptr, col, val, borrow=True)
    x = torch.randn(len(ptr) - 1, dtype=torch.float64, device="cuda")
    y = A.spmv(x)
    val *= 2.0
    torch.cuda.synchronize()
    assert torch.equal(A.spmv(x), 2.0 * y)
    A.close()
