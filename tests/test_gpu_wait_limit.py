"""The bound on the waits of on-chip solves (ks_ctx_set_wait_limit): which way
a solve takes.  A solve with one launch per operation counts launches of the
vector updates ("axpy"), an on-chip solve has none of its own."""
import numpy as np
import pytest

from tests import _problems as P

pytestmark = pytest.mark.gpu

DEFAULT = 1 << 21


@pytest.fixture
def limits(ctx):
    yield ctx.set_wait_limit
    ctx.set_wait_limit(DEFAULT)


def _launched(r):
    return r["prof"].get("axpy", {}).get("launches", 0)


def _system(n):
    # diagonally dominant and symmetric: tens of steps at any n
    rows = [[c for c in (i - 1, i, i + 1) if 0 <= c < n] for i in range(n)]
    col = np.array([c for r in rows for c in r], np.int32)
    ptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    val = np.where(col == np.repeat(np.arange(n), np.diff(ptr)), 3.0, -1.0)
    return ptr, col, val, np.random.default_rng(61).uniform(-1, 1, n)


@pytest.mark.parametrize("outer", ["cg", "bicg"])
@pytest.mark.parametrize("n", [1, 2, 511, 512, 513, 5000])
def test_limit_zero_takes_one_launch_per_operation(ctx, limits, n, outer):
    # also where one workgroup holds the system and would wait for nobody
    from solver_cpp_amd import api
    ptr, col, val, b = _system(n)
    A = api.Matrix(ctx, ptr, col, val, transpose=True)
    kw = dict(outer_eps=1e-12, outer_maxloop=500)
    for limit in (DEFAULT, 0, 1 << 30):
        limits(limit)
        x, r, _ = api.solve(ctx, A, b, outer, **kw)
        assert r["status"] == 0 and (_launched(r) > 0) == (limit == 0)
    A.close()


@pytest.mark.parametrize("outer,inner,kw", [
    ("cg", "NO", {}), ("bicg", "NO", {}),
    ("vpcg", "cg", dict(inner_maxloop=10, inner_precision=32)),
    ("vpgmres", "bicg", dict(outer_restart=20, inner_maxloop=10, inner_precision=32)),
])
def test_a_wait_that_runs_out_is_remembered(outer, inner, kw):
    # two polls are not enough for 256 workgroups: the solve is repeated by
    # launches, and the next ones are not tried on chip until the pause of 64
    # solves is over or a new limit is set
    from solver_cpp_amd import api
    ctx = api.Context(0)
    ptr, col, val, b = _system(256 * 512)
    A = api.Matrix(ctx, ptr, col, val, fp32=True, spd=True, transpose=True)

    def solve():
        x, r, _ = api.solve(ctx, A, b, outer, inner, history=False, outer_eps=1e-12, outer_maxloop=500, **kw)
        assert r["status"] == 0
        return x, r

    def counts():
        return tuple(ctx.on_chip().values())
    ctx.set_wait_limit(0)
    ref, r0 = solve()
    assert counts() == (0, 0)
    ctx.set_wait_limit(1)
    for k in range(65):
        x, r = solve()
        assert np.array_equal(x, ref) and r["iters"] == r0["iters"] and counts() == (1, 1)
    x, r = solve()
    assert np.array_equal(x, ref) and counts() == (2, 2)
    x, r = solve()  # pausing again
    assert counts() == (2, 2)
    ctx.set_wait_limit(DEFAULT)
    x, r = solve()
    assert counts() == (3, 2)
    assert np.linalg.norm(x - ref) <= 1e-9 * np.linalg.norm(ref)
    A.close()
    ctx.close()


def test_noalloc_solve_remembers_too(ctx, limits):
    import ctypes as C
    import torch
    from solver_cpp_amd import _abi, api
    ptr, col, val, b = _system(256 * 512)
    A = api.Matrix(ctx, ptr, col, val)
    bd = torch.from_numpy(b).cuda()
    p = _abi.make_params("cg", "NO", outer_eps=1e-12, outer_maxloop=500)
    p.flags |= _abi.KS_PTR_DEVICE
    out = []
    for limit in (0, 1):
        limits(limit)
        before = ctx.on_chip()
        for _ in range(3):
            x = torch.zeros_like(bd)
            torch.cuda.synchronize()
            res = _abi.KsResult()
            assert ctx.lib.ks_solve_noalloc(ctx.h, A.h, C.byref(p), bd.data_ptr(), x.data_ptr(), C.byref(res)) == 0
            assert res.status == 0
            out.append(x)
        assert ctx.on_chip()["solves"] - before["solves"] == limit  # one try in three solves
    assert all(torch.equal(x, out[0]) for x in out)
    A.close()
