"""The shape lookup of a small table (no GPU)."""
import pytest

from gpu_cc_tb_amd import SCHEMES
from gpu_cc_tb_amd import autotune as at


@pytest.mark.parametrize("read_ratio", [0.5, 1.0])
@pytest.mark.parametrize("scheme", ["tpl_nw", "tpl_wd"])
def test_small_table(scheme, read_ratio):
    """Below SMALL_TABLE rows 2PL at low skew runs the shape of theta 0.6; from
    there on, and where the rows are not given, the entry of its own bucket."""
    own, small = at.lookup(scheme, 0.1, read_ratio), at.lookup(scheme, 0.6, read_ratio)
    assert own != small
    assert at.lookup(scheme, 0.1, read_ratio, rows=at.SMALL_TABLE - 1) == small
    assert at.lookup(scheme, 0.1, read_ratio, rows=at.SMALL_TABLE) == own


def test_rows_change_nothing_else():
    for scheme in SCHEMES:
        for theta in (0.1, 0.6, 0.99):
            for rr in (0.5, 0.9, 1.0):
                if scheme in ("tpl_nw", "tpl_wd") and theta == 0.1 and rr != 0.9:
                    continue
                assert at.lookup(scheme, theta, rr, rows=4096) == at.lookup(scheme, theta, rr)
        assert at.lookup(scheme, 0.1, 0.5, key="stream", rows=4096) == at.lookup(scheme, 0.1, 0.5, key="stream")
