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
