"""The kernel names that bench.py reports for the stages are kernels of the library."""

import os
import re
import sys

import pytest

from gradwave_amd import _lib as L

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, REPO)

import bench  # noqa: E402


def _kernels():
    text = ""
    for name in os.listdir(os.path.join(REPO, "gradwave_amd", "csrc")):
        text += open(os.path.join(REPO, "gradwave_amd", "csrc", name)).read()
    found = re.findall(r"^(k_\w+)\(|__global__[^;{]*?\b(k_\w+)\(", text, flags=re.M)
    return {a or b for a, b in found}


@pytest.mark.skipif(not os.path.exists(L.LIB_PATH), reason="library not built")
@pytest.mark.parametrize("shape,planes", [((120, 120, 120), "k_plane_inv_w"), ((90, 90, 90), "k_plane_inv_w"),
                                          ((36, 36, 36), "k_plane_inv_any"), ((35, 70, 98), "k_plane_inv_any"),
                                          ((14, 24, 30), "k_plane_inv")])
def test_stage_kernels_exist(shape, planes):
    known = _kernels()
    assert {"k_plane_inv_w", "k_cgemm_inner", "k_dmul"} <= known
    fused = 1 if 14 in shape else 2
    lib = L.lib()
    try:
        for tile in range(14):
            for prec in (L.GW_FP64, L.GW_FP32):
                L.check(lib.gw_tune_set(L.GW_TUNE_GEMM_TILE, prec, tile), "gw_tune_set")
            for real in ("double", "float"):
                names = {s: re.split(r"[<( ]", bench.stage_kernel(s, real, shape, fused))[0] for s in L.STAGES}
                assert set(names.values()) <= known, names
                assert names["plane_inv"] == planes
                assert names["becp"] == ("k_gemm_inner_tile" if 1 <= tile <= 5 else "k_cgemm_inner")
                # three products per complex one: the explicit variants only
                assert bench.gemm_mfma_fraction("becp", real) == (0.75 if tile >= 10 else 1.0)
    finally:
        for prec in (L.GW_FP64, L.GW_FP32):
            L.check(lib.gw_tune_set(L.GW_TUNE_GEMM_TILE, prec, 0), "gw_tune_set")
