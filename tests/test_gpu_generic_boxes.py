"""The generic box FFT kernels where they run by default: boxes with a length below 15 or
above 160 (and 168, 180, 192, ... with a two-codelet split), whose x-planes fit LDS or are
split into stick and column kernels, against the oracle's apply (core/batch.py:405-505)
and density (core/batch.py:562-587); and by option (GW_PLAN_LEGACY) on boxes that take the
wave lines otherwise."""

import pytest
import torch

from gpu_cases import dev, rand_block, ref_h, say
from test_gpu_box_lengths import _check_apply, _gpu_h, _rel, _si2

pytestmark = pytest.mark.gpu

from gradwave_amd import _lib as L  # noqa: E402

# (shape, fused_planes FP64, FP32): 1 plane in LDS, 0 split
_DEFAULT = [((14, 24, 30), 1, 1), ((24, 12, 36), 1, 1), ((25, 30, 168), 1, 1), ((180, 18, 24), 1, 1),
            ((20, 192, 21), 1, 1), ((16, 196, 15), 1, 1), ((27, 16, 210), 1, 1), ((224, 15, 18), 1, 1),
            ((18, 225, 16), 1, 1), ((240, 16, 21), 1, 1), ((15, 24, 256), 1, 1), ((14, 108, 105), 0, 1),
            ((12, 168, 160), 0, 0)]


@pytest.mark.parametrize("shape,f64,f32", _DEFAULT)
def test_default_boxes_of_the_generic_kernels(shape, f64, f32):
    say(f"generic box {shape}")
    s = _si2(shape)
    cpu, _, h = _gpu_h(s, toeplitz="off")
    assert (h.info()["fused_planes"], h.info(torch.complex64)["fused_planes"]) == (f64, f32)
    assert h.local_path == "fft"
    _check_apply(s, h, cpu, seed=101)


@pytest.mark.parametrize("shape,f64,f32", [((24, 30, 36), 1, 1), ((36, 24, 30), 1, 1), ((30, 36, 24), 1, 1),
                                           ((24, 120, 96), 0, 1), ((36, 36, 36), 1, 1)])
def test_generic_kernels_on_request(shape, f64, f32):
    """Wave-line boxes with GW_PLAN_LEGACY: the plane kernels of FP64 x-planes above the
    LDS budget are split, and so are all with GW_PLAN_FORCE_UNFUSED."""
    s = _si2(shape)
    cpu, _, h = _gpu_h(s, toeplitz="off")
    for flags in (L.GW_PLAN_LEGACY, L.GW_PLAN_LEGACY | L.GW_PLAN_FORCE_UNFUSED):
        say(f"generic kernels {shape} flags {flags}")
        h.set_flags(flags)
        want = (0, 0) if flags & L.GW_PLAN_FORCE_UNFUSED else (f64, f32)
        assert (h.info()["fused_planes"], h.info(torch.complex64)["fused_planes"]) == want
        _check_apply(s, h, cpu, seed=102)


@pytest.mark.parametrize("shape", [(14, 24, 30), (20, 25, 168), (14, 108, 105)])
def test_density_on_generic_boxes(shape):
    from gradwave_amd.hamiltonian import density_b
    from oracle.hamiltonian import density_b as ref_density

    say(f"density on a generic box {shape}")
    s = _si2(shape)
    cpu, gpu, _ = _gpu_h(s, toeplitz="off")
    c = rand_block(cpu.nk, 5, cpu.npw_max, cpu.mask, seed=103)
    g = torch.Generator().manual_seed(104)
    occ = torch.rand(cpu.nk, 5, dtype=torch.float64, generator=g)
    kw = torch.rand(cpu.nk, dtype=torch.float64, generator=g)
    want = ref_density(c, occ, kw, cpu, s.shape, s.grid.volume)
    for dtype, tol in ((torch.complex128, 1e-12), (torch.complex64, 2e-5)):
        got = density_b(c.to(dev(), dtype), occ.to(dev()), kw.to(dev()), gpu, s.shape, s.grid.volume)
        assert _rel(got.cpu(), want) < tol
