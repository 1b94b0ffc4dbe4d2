"""GMRES's one-workgroup steps (projection finisher with the norm step beside
it, back substitution) over the column counts at which they change, against
the lanes-per-row kernels, whose projection, norm and rotations run apart.

The residual stays above 1e-3 here, so classical Gram-Schmidt keeps the basis
orthogonal to rounding and the two histories differ by rounding times at most
the steps' growth: 1e-7 relative is allowed, and 1e-7 of x."""
import numpy as np
import pytest

from tests import _problems as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("restart", [2, 3, 9, 10, 17, 18, 33, 34, 64, 65, 66, 80])
def test_restarts(ctx, restart):
    from solver_cpp_amd import api
    ptr, col, val = P.poisson2d(96)[:3]
    b = np.random.default_rng(11).uniform(-1, 1, len(ptr) - 1)
    out = []
    for layout in ("auto", "vector"):
        A = api.Matrix(ctx, ptr, col, val, layout=layout)
        # ends inside the second cycle
        out.append(api.solve(ctx, A, b, "gmres", outer_eps=0.0, outer_restart=restart,
                             outer_maxloop=restart + max(1, restart // 2)))
        A.close()
    (x, r, h), (y, s, g) = out
    assert r["status"] == s["status"] == 2 and r["iters"] == s["iters"] and h.shape == g.shape
    assert h[-1, 1] > 1e-3 and np.allclose(h, g, rtol=1e-7)
    assert np.linalg.norm(x - y) <= 1e-7 * np.linalg.norm(y)
