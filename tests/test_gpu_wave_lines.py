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
