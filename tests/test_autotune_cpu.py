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


@built
def test_saved_file_leaves_the_tiles_to_the_rule(tmp_path):
    """A file that the library loads by itself sets what holds for any program; one GEMM
    tile for every size (three products among them) takes a call of the program's own."""
    path = tmp_path / "tune.json"
    path.write_text(json.dumps({"gemm_tile": {"fp64": 12, "fp32": 13}, "gemm_tile_combine": {"fp64": 11, "fp32": 4},
                                "radix": {"24": 4}, "gemm_wgs": 1024, "xpass": {"fp64": 208, "fp32": 10408},
                                "plane_bands": {"fp64": [2, 1], "fp32": [4, 2]}}))
    code = """
from gradwave_amd import _lib as L, autotune
g = L.lib().gw_tune_get
def tiles():
    return [g(L.GW_TUNE_GEMM_TILE, p + 256 * op) for op in (1, 2) for p in (L.GW_FP64, L.GW_FP32)]
def rest():
    return [g(L.GW_TUNE_RADIX, 24), g(L.GW_TUNE_GEMM_WGS, 0), g(L.GW_TUNE_XPASS, L.GW_FP64),
            g(L.GW_TUNE_PLANE_BANDS, L.GW_FP32 + 256)]
print(tiles(), rest())
autotune.load()
print(tiles(), rest())
"""
    r = subprocess.run([sys.executable, "-c", code], cwd=REPO, env={**os.environ, "GW_TUNE_FILE": str(path)},
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    assert r.stdout.split("\n")[:2] == ["[0, 0, 0, 0] [4, 1024, 208, 4]", "[12, 13, 11, 4] [4, 1024, 208, 4]"]
