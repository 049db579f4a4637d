"""The wave-line passes of the local term in the launch forms that large blocks take
(staged tiles, several bands per workgroup), on every box length they are built for.
A transform rounds alike in every form, so a large block of repeated bands equals the
same bands in a small one to the bit; the small one is checked against the oracle's
apply (core/batch.py:405-505)."""

import pytest
import torch

from gpu_cases import dev, rand_block, ref_h, say
from test_gpu_box_lengths import _SYS, _WAVE_LENGTHS, _gpu_h, _rel, _si2

pytestmark = pytest.mark.gpu

from gradwave_amd import _lib as L  # noqa: E402

_BANDS = 5


def _repeated(c, nb):
    return c[:, torch.arange(nb) % c.shape[1]].contiguous()


@pytest.mark.parametrize("n", _WAVE_LENGTHS)
def test_x_pass_of_large_blocks_matches_small_ones(n):
    """Blocks of enough bands for 8 (FP32 also 16) bands per workgroup: FP32 moves
    staged pairs where n2 n3 is even, odd n included, and reads lines straight from
    the box where it is odd; small blocks take one band per workgroup."""
    for shape in ((n, 15, 20), (n, 15, 21)):
        s = _si2(shape)
        cpu, _, h = _gpu_h(s, toeplitz="off")
        c = rand_block(cpu.nk, _BANDS, cpu.npw_max, cpu.mask, seed=n)
        want = ref_h(s).apply(c)
        # a workgroup's four waves take at most 64 lines, and 2048 workgroups are aimed at
        nb = 8 * 2048 * 64 // (shape[1] * shape[2] * cpu.nk) + 3
        for dtype, tol in ((torch.complex128, 1e-12), (torch.complex64, 2e-5)):
            say(f"x pass of {nb} bands {shape} {dtype}")
            few = c.to(dev(), dtype)
            many = _repeated(few, nb)
            terms = L.GW_TERM_KINETIC | L.GW_TERM_LOCAL
            got = h.apply_terms(many, terms)
            assert torch.equal(got, _repeated(h.apply_terms(few, terms), nb))
            assert _rel(h.apply(many)[:, :_BANDS].cpu().to(torch.complex128), want) < tol
        _SYS.pop(shape)


# y and z lines of every class of the plane kernels (largest part count 8, 10, 16)
@pytest.mark.parametrize("shape", [(18, 24, 35), (20, 27, 64), (16, 90, 28), (21, 32, 100), (15, 75, 30), (18, 28, 160)])
@pytest.mark.parametrize("dtype", [torch.complex128, torch.complex64])
def test_planes_with_several_bands_per_item(shape, dtype):
    """GW_TUNE_PLANE_BANDS 3 over 8 bands (the last item part-full) equals one band per
    item to the bit, sphere padding included."""
    s = _si2(shape)
    cpu, _, h = _gpu_h(s, toeplitz="off")
    assert h.info(dtype)["fused_planes"] == 2
    say(f"plane bands {shape} {dtype}")
    c = rand_block(cpu.nk, 8, cpu.npw_max, cpu.mask, seed=95).to(dev(), dtype)
    terms, prec, lib = L.GW_TERM_KINETIC | L.GW_TERM_LOCAL, L.precision_of(dtype), L.lib()
    try:
        L.check(lib.gw_tune_set(L.GW_TUNE_PLANE_BANDS, prec, 1), "gw_tune_set")
        one = h.apply_terms(c, terms)
        L.check(lib.gw_tune_set(L.GW_TUNE_PLANE_BANDS, prec, 3), "gw_tune_set")
        three = h.apply_terms(c, terms)
    finally:
        L.check(lib.gw_tune_set(L.GW_TUNE_PLANE_BANDS, prec, 0), "gw_tune_set")
    assert torch.equal(three, one)
    assert _rel(h.apply(c)[:, :3].cpu().to(torch.complex128), ref_h(s).apply(c[:, :3].cpu().to(torch.complex128))) < (
        1e-12 if dtype == torch.complex128 else 2e-5)


def _batch(shapes, flags=0):
    from gradwave_amd.batching import RaggedBatch

    hams, blocks, wants = [], [], []
    for i, shape in enumerate(shapes):
        s = _si2(shape)
        cpu, _, h = _gpu_h(s, toeplitz="off", flags=flags)
        c = rand_block(cpu.nk, 9 + i, cpu.npw_max, cpu.mask, seed=96 + i)
        hams.append(h)
        blocks.append(c)
        wants.append(ref_h(s).apply(c))
    return RaggedBatch(hams), hams, blocks, wants


@pytest.mark.parametrize("shapes,fused", [
    (((24, 30, 36), (112, 16, 27), (15, 75, 30), (20, 18, 160)), (2, 2, 2, 2)),  # parts up to 16
    (((24, 30, 36), (14, 24, 30), (36, 36, 36)), (2, 1, 2)),                      # one cell without wave lines
    (((14, 24, 30), (20, 25, 168)), (1, 1)),                                      # none with them
])
def test_ragged_batches_of_every_class(shapes, fused):
    """The ragged wave-line passes of large part counts, and the generic passes that a
    batch takes as a whole when a cell of it has no wave lines."""
    batch, hams, blocks, wants = _batch(shapes)
    for dtype, tol in ((torch.complex128, 1e-12), (torch.complex64, 2e-5)):
        say(f"ragged batch {shapes} {dtype}")
        assert tuple(h.info(dtype)["fused_planes"] for h in hams) == fused
        for o, w in zip(batch.apply([c.to(dev(), dtype) for c in blocks]), wants):
            assert _rel(o.cpu().to(torch.complex128), w) < tol


@pytest.mark.parametrize("shape", [(24, 24, 24), (36, 36, 36), (18, 24, 35), (20, 27, 64), (35, 70, 98), (21, 32, 100),
                                   (72, 24, 72), (18, 28, 160)])
@pytest.mark.parametrize("dtype", [torch.complex128, torch.complex64])
def test_kinetic_term_is_rounded_once(shape, dtype):
    """t c + V psi with V = 1 and t a thousand times as large: the result is within one
    rounding of the exact sum, with a tenth of one for the local part (its transforms'
    error, some ten roundings, a thousandth of the whole), so t c is not rounded by itself."""
    import numpy as np

    say(f"kinetic rounding {shape} {dtype}")
    s = _si2(shape)
    cpu, gpu, h = _gpu_h(s, toeplitz="off")
    g = torch.Generator().manual_seed(97)
    u = 2.0 ** (-53 if dtype == torch.complex128 else -24)
    rdt = torch.float64 if dtype == torch.complex128 else torch.float32
    t = (1000.0 * (1.0 + torch.rand(cpu.nk, cpu.npw_max, dtype=torch.float64, generator=g))).to(rdt).double()
    h.plan.set_potential(torch.ones(shape, dtype=torch.float64, device=dev()))
    h.plan.set_kinetic(t.to(dev()))
    part = [(1.0 + torch.rand(cpu.nk, 9, cpu.npw_max, dtype=torch.float64, generator=g)).to(rdt) for _ in range(2)]
    c = torch.complex(*part).to(dtype) * cpu.mask[:, None, :]
    terms, prec, lib = L.GW_TERM_KINETIC | L.GW_TERM_LOCAL, L.precision_of(dtype), L.lib()
    for bands in (1, 4):
        try:
            L.check(lib.gw_tune_set(L.GW_TUNE_PLANE_BANDS, prec, bands), "gw_tune_set")
            got = h.apply_terms(c.to(dev()), terms).cpu()
        finally:
            L.check(lib.gw_tune_set(L.GW_TUNE_PLANE_BANDS, prec, 0), "gw_tune_set")
        for have, x in ((got.real, c.real), (got.imag, c.imag)):
            want = x.numpy().astype(np.longdouble) * (t[:, None, :].numpy().astype(np.longdouble) + 1)
            err = np.abs(have.numpy().astype(np.longdouble) - want)
            assert bool((err <= 1.1 * u * want).all()), float((err / np.maximum(u * want, 1e-300)).max())
