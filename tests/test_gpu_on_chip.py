"""On-chip solves (many steps per launch, workgroups that wait for each other)
against the same solve with one launch per operation, which a wait limit of 0
takes: sizes at the edges of a workgroup, of the rows per thread and of the
range, ends of launches, and the ways a solve can end.

The two sum their dot products in different orders, so a dot of n products
differs by at most about n eps of its absolute sum; over the steps of these
well-conditioned solves x stays within 1e-9 of the other path's, relative, at
a tolerance of 1e-12, and the step counts within one."""
import threading

import numpy as np
import pytest

from tests import _problems as P

pytestmark = pytest.mark.gpu

WG = 512  # rows of a workgroup at one row per thread


def _tridiag(n, seed=5):
    # diagonally dominant, condition number below 20: tens of steps at any n
    rng = np.random.default_rng(seed)
    i = np.arange(n)
    rows = np.concatenate([i[1:], i, i[:-1]])
    cols = np.concatenate([i[:-1], i, i[1:]])
    vals = np.concatenate([np.full(n - 1, -1.0), 2.5 + rng.random(n), np.full(n - 1, -1.0)])
    o = np.lexsort((cols, rows))
    ptr = np.zeros(n + 1, np.int32)
    ptr[1:] = np.cumsum(np.bincount(rows, minlength=n))
    return ptr, cols[o].astype(np.int32), vals[o], rng.uniform(-1, 1, n)


@pytest.fixture
def both(ctx):
    from solver_cpp_amd import api

    def run(A, b, *args, **kw):
        out = []
        try:
            for limit in (1 << 21, 0):
                ctx.set_wait_limit(limit)
                out.append(api.solve(ctx, A, b, *args, **kw))
        finally:
            ctx.set_wait_limit(1 << 21)
        return out
    return run


SOLVERS = [("cg", "NO", {}), ("vpcg", "cg", dict(inner_maxloop=10, inner_precision=32)),
           ("vpcg", "cg", dict(inner_maxloop=10, inner_precision=64))]


def _same(one, two, tol=1e-9):
    (x, r, h), (y, s, g) = one, two
    assert r["status"] == s["status"] == 0 and abs(r["iters"] - s["iters"]) <= 1
    assert np.linalg.norm(x - y) <= tol * np.linalg.norm(y)
    m = min(len(h), len(g))
    assert abs(len(h) - len(g)) <= 1 and np.array_equal(h[:m, 0], g[:m, 0])
    assert r["steps"] + 1 >= s["steps"] and abs(r["spmv"] - s["spmv"]) <= 2 + abs(r["iters"] - s["iters"]) * 100


@pytest.mark.parametrize("outer,inner,kw", SOLVERS)
@pytest.mark.parametrize("n", [1, 2, WG - 1, WG, WG + 1, 64 * WG + 3, 256 * WG, 256 * WG + 1, 512 * WG + 1,
                               1024 * WG - 1, 1024 * WG, 1024 * WG + 1])
def test_sizes(ctx, both, n, outer, inner, kw):
    from solver_cpp_amd import api
    ptr, col, val, b = _tridiag(n)
    A = api.Matrix(ctx, ptr, col, val, fp32=True, spd=True, transpose=True)
    _same(*both(A, b, outer, inner, outer_eps=1e-12, outer_maxloop=500, **kw))
    A.close()


@pytest.mark.parametrize("outer,inner,kw", SOLVERS)
def test_stencils(ctx, both, outer, inner, kw):
    # 5- and 7-point rows, every neighbour of some row in another workgroup
    from solver_cpp_amd import api
    for ptr, col, val in (P.poisson2d(77)[:3], P.convdiff3d(23, pe=0.0)[:3]):
        b = np.random.default_rng(3).uniform(-1, 1, len(ptr) - 1)
        A = api.Matrix(ctx, ptr, col, val, fp32=True, spd=True, transpose=True)
        _same(*both(A, b, outer, inner, outer_eps=1e-12, outer_maxloop=5000, **kw))
        A.close()


def test_run_to_run_and_index_formats(ctx):
    from solver_cpp_amd import api
    ptr, col, val = P.poisson2d(150)[:3]
    b = np.random.default_rng(4).uniform(-1, 1, len(ptr) - 1)
    ref = None
    for layout in ("auto", "auto", "delta", "col32"):
        A = api.Matrix(ctx, ptr, col, val, layout=layout)
        x, r, h = api.solve(ctx, A, b, "cg", outer_eps=1e-12, outer_maxloop=5000)
        assert r["status"] == 0
        ref = ref or (x, h)
        assert np.array_equal(x, ref[0]) and np.array_equal(h, ref[1])
        A.close()


@pytest.mark.parametrize("maxloop", [1, 2, 7, 1023, 1024, 1025, 2048, 2049])
def test_cg_ends_at_maxloop(ctx, both, maxloop):
    # the limit inside a launch of 1024 steps, at its end and one past it; the
    # history entry for entry while it lasts (a residual that stagnates in
    # rounding differs between the paths: only its place is compared)
    from solver_cpp_amd import api
    ptr, col, val = P.poisson2d(24)[:3]
    b = np.random.default_rng(6).uniform(-1, 1, len(ptr) - 1)
    A = api.Matrix(ctx, ptr, col, val)
    (x, r, h), (y, s, g) = both(A, b, "cg", outer_eps=0.0, outer_maxloop=maxloop)
    if s["status"] == 2:
        assert r["status"] == 2 and r["iters"] == s["iters"] == maxloop + 1 and r["n_hist"] == s["n_hist"] == maxloop
    m = min(40, len(h), len(g))
    assert np.array_equal(h[:m, 0], g[:m, 0]) and np.allclose(h[:m, 1], g[:m, 1], rtol=1e-6)
    A.close()


@pytest.mark.parametrize("g", [60, 160])
def test_cg_ill_conditioned(ctx, both, g):
    # log-normal coefficients (condition number up to about 1e6): hundreds of
    # steps and, at 160, three launches or more.  Rounding moves the step count
    # here, so each path is held to the tolerance itself and the two solutions
    # to condition number times the residuals
    from solver_cpp_amd import api
    ptr, col, val = P.aniso(g)[:3]
    b = np.random.default_rng(7).uniform(-1, 1, len(ptr) - 1)
    A = api.Matrix(ctx, ptr, col, val)
    one, two = both(A, b, "cg", outer_eps=1e-11, outer_maxloop=20000)
    assert g == 60 or one[1]["iters"] > 2048
    for x, r, h in (one, two):
        assert r["status"] == 0 and r["relres_true"] <= 2e-11 and r["n_hist"] == r["iters"]
    assert np.linalg.norm(one[0] - two[0]) <= 1e6 * 4e-11 * np.linalg.norm(two[0])
    A.close()


@pytest.mark.parametrize("outer,inner,kw", SOLVERS)
def test_zero_and_nonfinite_right_sides(ctx, both, outer, inner, kw):
    from solver_cpp_amd import api
    ptr, col, val, b = _tridiag(3 * WG)
    A = api.Matrix(ctx, ptr, col, val, fp32=True, spd=True, transpose=True)
    for v in (0.0, np.nan, np.inf):
        c = np.zeros_like(b)
        c[700] = v
        (x, r, _), (y, s, _) = both(A, c, outer, inner, outer_eps=1e-10, outer_maxloop=30, **kw)
        assert r["status"] == s["status"] and r["iters"] == s["iters"]
        if v == 0.0:
            assert r["status"] == 0 and not x.any()
    A.close()


@pytest.mark.parametrize("outer,inner,kw", SOLVERS)
def test_initial_guess(ctx, both, outer, inner, kw):
    from solver_cpp_amd import api
    ptr, col, val, b = _tridiag(5 * WG + 17)
    A = api.Matrix(ctx, ptr, col, val, fp32=True, spd=True, transpose=True)
    x0 = np.random.default_rng(8).standard_normal(len(b))
    _same(*both(A, b, outer, inner, x0=x0, outer_eps=1e-12, outer_maxloop=500, **kw))
    A.close()


def test_two_threads(ctx):
    # two contexts solve at once: on-chip solves of one device take turns
    from solver_cpp_amd import api
    ptr, col, val = P.poisson2d(250)[:3]
    b = np.random.default_rng(9).uniform(-1, 1, len(ptr) - 1)
    kw = dict(outer_eps=1e-12, outer_maxloop=5000)
    A = api.Matrix(ctx, ptr, col, val)
    ref = api.solve(ctx, A, b, "cg", **kw)[0]
    A.close()
    got = [None] * 3

    def work(k):
        c = api.Context(0)
        M = api.Matrix(c, ptr, col, val)
        got[k] = [api.solve(c, M, b, "cg", **kw)[0] for _ in range(4)]
        M.close()
        c.close()
    ts = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert all(np.array_equal(x, ref) for xs in got for x in xs)


# BiCG holds A and A^T: in FP64 at most two rows per thread
BICG = [("bicg", "NO", {}), ("vpgmres", "bicg", dict(outer_restart=20, inner_maxloop=10, inner_precision=32))]


def _upwind(n, seed=12):
    # nonsymmetric, diagonally dominant by rows and columns
    ptr, col, val, b = _tridiag(n, seed)
    row = np.repeat(np.arange(n), np.diff(ptr))
    return ptr, col, np.where(col < row, 1.1 * val, val), b


@pytest.mark.parametrize("outer,inner,kw", BICG)
@pytest.mark.parametrize("n", [1, 2, WG - 1, WG + 1, 64 * WG + 3, 256 * WG, 256 * WG + 1, 512 * WG, 512 * WG + 1,
                               1024 * WG + 1])
def test_bicg_sizes(ctx, both, n, outer, inner, kw):
    from solver_cpp_amd import api
    ptr, col, val, b = _upwind(n)
    A = api.Matrix(ctx, ptr, col, val, fp32=True, transpose=True)
    _same(*both(A, b, outer, inner, outer_eps=1e-12, outer_maxloop=500, **kw))
    x0 = np.random.default_rng(13).standard_normal(n)
    _same(*both(A, b, outer, inner, x0=x0, outer_eps=1e-12, outer_maxloop=500, **kw))
    A.close()


@pytest.mark.parametrize("outer,inner,kw", BICG)
def test_bicg_stencil_and_right_sides(ctx, both, outer, inner, kw):
    # 7-point upwind rows with neighbours in other workgroups; b of zeros, NaN and Inf
    from solver_cpp_amd import api
    ptr, col, val = P.convdiff3d(17, pe=0.8)[:3]
    val = np.where(col == np.repeat(np.arange(len(ptr) - 1), np.diff(ptr)), val + 2.0, val)
    b = np.random.default_rng(14).uniform(-1, 1, len(ptr) - 1)
    A = api.Matrix(ctx, ptr, col, val, fp32=True, transpose=True)
    _same(*both(A, b, outer, inner, outer_eps=1e-12, outer_maxloop=500, **kw))
    for v in (0.0, np.nan, np.inf):
        c = np.zeros_like(b)
        c[700] = v
        (x, r, _), (y, s, _) = both(A, c, outer, inner, outer_eps=1e-10, outer_maxloop=30, **kw)
        assert r["status"] == s["status"] and r["iters"] == s["iters"]
    A.close()


@pytest.mark.parametrize("maxloop", [1, 2, 1023, 1024, 1025, 2049])
def test_bicg_ends_at_maxloop(ctx, both, maxloop):
    from solver_cpp_amd import api
    ptr, col, val, b = _upwind(3 * WG)
    A = api.Matrix(ctx, ptr, col, val, transpose=True)
    (x, r, h), (y, s, g) = both(A, b, "bicg", outer_eps=0.0, outer_maxloop=maxloop)
    if s["status"] == 2 and r["status"] == 2:
        assert r["iters"] == s["iters"] == maxloop + 1 and r["n_hist"] == s["n_hist"] == maxloop
    m = min(10, len(h), len(g))
    assert np.array_equal(h[:m, 0], g[:m, 0]) and np.allclose(h[:m, 1], g[:m, 1], rtol=1e-6)
    A.close()
