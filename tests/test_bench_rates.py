"""bench.py's rates: the roofline kernel's fraction of the measured read rate is
the rate that its `achieved` field reports."""
import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))


class _Stream:
    def stream_rate(self, kind):
        return {"read": 7000.0, "copy": 6000.0}[kind]


@pytest.mark.parametrize("achieved,frac", [(3500.0, 0.5), (None, None)])
def test_ceiling_is_of_the_achieved_rate(achieved, frac):
    import bench
    out = bench.hbm_ceiling(_Stream(), achieved)
    assert out.get("roofline_achieved_frac_of_read") == frac
    assert out["read_GBps"] == 7000.0 and out["copy_GBps"] == 6000.0
    assert not [k for k in out if "format" in k]
