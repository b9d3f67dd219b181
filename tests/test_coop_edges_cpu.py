"""Where a small layer with row scales is one launch: the edges of the rule on both sides."""
import pytest


@pytest.mark.parametrize("Q, d, R, served", [(77, 1600, 4800, 1), (80, 1600, 4800, 1), (81, 1600, 4800, 0), (500, 192, 2000, 1), (512, 100, 2000, 1),
                                             (513, 100, 2000, 0), (550, 192, 2000, 0), (560, 100, 2000, 0)])
def test_row_scales(Q, d, R, served):
    from bsipytorch_amd import _lib

    assert _lib.lib.bsi_hip_linear_coop_serves(Q, d, R, 2, 7, _lib.LAYOUT_INT8, 6) == served
