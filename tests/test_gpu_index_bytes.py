"""ks_mat_index_bytes of matrices that are read as row patterns or row classes:
the entry format such a matrix would have, from what was stored at creation."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _band(n, offsets):
    # row i holds the entries i + d that fall inside [0, n)
    i = np.arange(n)[:, None] + np.array(sorted(offsets))[None, :]
    ok = (i >= 0) & (i < n)
    ptr = np.zeros(n + 1, np.int32)
    ptr[1:] = np.cumsum(ok.sum(1))
    return ptr, i[ok].astype(np.int32), (np.array(sorted(offsets))[None, :] + 0.5 + 0 * i)[ok]


@pytest.mark.parametrize("values", ["by_offset", "by_entry"])  # row classes, row patterns
@pytest.mark.parametrize("offsets,ib,ibt", [
    ([-32767, -3, 0, 1, 32767], 2, 2),   # int16 offsets
    ([-49152, -3, 0, 1, 49152], 2, 2),   # delta codes: the lowest first code
    ([-49153, -3, 0, 1, 49153], 4, 4),
    ([0, 65535], 2, 4), ([0, 65536], 4, 4),
    ([16383, 40000], 2, 2), ([16384, 40000], 4, 2),
])
def test_entry_format_of_patterns_and_classes(ctx, offsets, ib, ibt, values):
    from solver_cpp_amd import api
    n = 140_000
    ptr, col, val = _band(n, offsets)
    if values == "by_entry":
        val = np.random.default_rng(41).standard_normal(len(col))
    A = api.Matrix(ctx, ptr, col, val, transpose=True, fp32=True)
    assert A.spmv_bytes() == (17 * n if values == "by_offset" else 18 * n + 8 * len(col))
    for prec in (64, 32):
        assert A.index_bytes(False, prec) == ib and A.index_bytes(True, prec) == ibt
    A.update_values(np.random.default_rng(42).standard_normal(len(col)))  # ends the classes: patterns
    assert A.index_bytes(False) == ib and A.index_bytes(True) == ibt
    A.close()


@pytest.mark.parametrize("reverse", [False, True])
def test_unsorted_rows_have_no_delta_codes(ctx, reverse):
    from solver_cpp_amd import api
    ptr, col, val = _band(100_000, [-40000, -1, 0, 1, 40000])
    if reverse:
        for i in range(len(ptr) - 1):
            col[ptr[i]:ptr[i + 1]] = col[ptr[i]:ptr[i + 1]][::-1].copy()
            val[ptr[i]:ptr[i + 1]] = val[ptr[i]:ptr[i + 1]][::-1].copy()
    A = api.Matrix(ctx, ptr, col, val, transpose=True)
    assert A.index_bytes(False) == (4 if reverse else 2) and A.index_bytes(True) == 2
    A.close()


def test_asking_does_no_device_work(ctx):
    # a call of a few microseconds; building 20 million delta codes to look
    # whether they fit takes hundreds
    from solver_cpp_amd import api
    ptr, col, val = _band(4_000_000, [-40000, -1, 0, 1, 40000])
    A = api.Matrix(ctx, ptr, col, val)
    best = 1.0
    for _ in range(20):
        t = time.perf_counter()
        assert A.index_bytes() == 2
        best = min(best, time.perf_counter() - t)
    assert best < 30e-6, best
    A.close()
