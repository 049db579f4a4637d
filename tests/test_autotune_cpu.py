"""What the tuner may choose and what a saved file sets, without a GPU."""

import json
import os
import subprocess
import sys
from types import SimpleNamespace

import pytest

from gradwave_amd import _lib as L
from gradwave_amd import autotune

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
built = pytest.mark.skipif(not os.path.exists(L.LIB_PATH), reason="library not built")


@built
@pytest.mark.parametrize("n", [24, 36, 48])
def test_x_pass_shape_is_left_alone_where_it_has_no_effect(n):
    """Only the 90 and 120 cubes' kernels take GW_TUNE_XPASS; elsewhere every shape runs
    the same code, and a winner would be noise, kept for those cubes."""
    before = {name: L.lib().gw_tune_get(L.GW_TUNE_XPASS, prec) for name, prec in (("fp64", L.GW_FP64),
                                                                                  ("fp32", L.GW_FP32))}
    assert autotune.tune_xpass([SimpleNamespace(shape=(n, n, n))]) == before
