"""The V(r) adjoint of two operators on two streams at once, against the same calls in turn."""

from types import SimpleNamespace

import pytest
import torch

from gpu_cases import dev, rand_block, say
from test_gpu_box_lengths import _gpu_h, _si2

pytestmark = pytest.mark.gpu

from gradwave_amd import adjoint as A  # noqa: E402


def _problem(shape, nb, seed):
    s = _si2(shape)
    cpu, _, h = _gpu_h(s, toeplitz="off")
    c, g = (rand_block(cpu.nk, nb, cpu.npw_max, cpu.mask, seed=seed + i).to(dev()) for i in range(2))
    return SimpleNamespace(fwd=h, shape=s.shape), c, g


def test_v_adjoints_on_two_streams():
    say("V adjoint on two streams")
    problems = [_problem((30, 28, 27), 40, 90), _problem((36, 36, 36), 33, 92)]
    want = [A.adjoint_v(*p) for p in problems]
    streams = [torch.cuda.Stream() for _ in problems]
    torch.cuda.synchronize()
    got = [[], []]
    for _ in range(6):
        for i, (p, st) in enumerate(zip(problems, streams)):
            with torch.cuda.stream(st):
                got[i].append(A.adjoint_v(*p))
    torch.cuda.synchronize()
    for i, w in enumerate(want):
        assert all(torch.equal(x, w) for x in got[i])


@pytest.mark.parametrize("dtype,tol", [(torch.complex128, 1e-12), (torch.complex64, 1e-12)])
def test_v_adjoint_in_band_chunks(dtype, tol, monkeypatch):
    """Chunks sum in another order only (FP64 sums of the same products)."""
    from gradwave_amd import hamiltonian

    say(f"V adjoint in chunks {dtype}")
    op, c, g = _problem((30, 28, 27), 19, 94)
    c, g = c.to(dtype), g.to(dtype)
    whole = A.adjoint_v(op, c, g)
    calls = 2 * c.shape[0] * 19 * 30 * 28 * 27 * c.element_size()  # above the whole block's two boxes
    monkeypatch.setattr(hamiltonian, "_LIB_FFT_BUDGET_BYTES", calls // 7)
    parts = A.adjoint_v(op, c, g)
    assert float((parts - whole).abs().max() / whole.abs().max()) < tol
