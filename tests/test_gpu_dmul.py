"""The D multiply of the nonlocal term (core/batch.py:480-505): inside the split-K
reduction of the projection for narrow D, in its own kernel where a column of D has many
entries (each partial would be read once per entry), against the oracle's apply."""

from types import SimpleNamespace

import pytest
import torch

from gpu_cases import dev, rand_block, say, select_k
from test_gpu_box_lengths import _rel, _si2

pytestmark = pytest.mark.gpu

from gradwave_amd import _lib as L  # noqa: E402
from gradwave_amd.hamiltonian import BatchedHamiltonian  # noqa: E402
from oracle.hamiltonian import BatchedHamiltonian as RefH  # noqa: E402
from oracle.hamiltonian import BatchedK  # noqa: E402


def _case(nproj, dij, nb):
    s = _si2((20, 18, 21))
    cpu, gpu, _ = select_k(s)
    g = torch.Generator().manual_seed(70)
    p = torch.randn(cpu.nk, nproj, cpu.npw_max, dtype=torch.complex128, generator=g) * cpu.mask[:, None, :]
    c = rand_block(cpu.nk, nb, cpu.npw_max, cpu.mask, seed=71)
    want = RefH(BatchedK(npw=cpu.npw, mask=cpu.mask, flat_idx=cpu.flat_idx, kpg=cpu.kpg, t=cpu.t, proj_phase_free=p,
                         proj_atom_index=cpu.proj_atom_index, dij_full=dij), s.shape, s.v_r, p).apply(c)
    bk = SimpleNamespace(npw=gpu.npw, mask=gpu.mask, flat_idx=gpu.flat_idx, t=gpu.t, dij_full=dij.to(dev()))
    return BatchedHamiltonian(bk, s.shape, s.v_r.to(dev()), p.to(dev()), toeplitz="off"), c, want


@pytest.mark.parametrize("dtype,tol", [(torch.complex128, 1e-12), (torch.complex64, 2e-5)])
@pytest.mark.parametrize("kind,apart", [("zero", False), ("diagonal", False), ("pairs", False), ("column", True),
                                        ("dense", True)])
def test_d_multiply_by_the_width_of_d(kind, apart, dtype, tol):
    nproj, nb = 64, 7
    g = torch.Generator().manual_seed(72)
    dij = torch.zeros(nproj, nproj, dtype=torch.float64)
    r = torch.randn(nproj, nproj, dtype=torch.float64, generator=g)
    if kind == "diagonal":
        dij = torch.diag(r.diagonal())
    elif kind == "pairs":
        dij = r * torch.block_diag(*[torch.ones(2, 2, dtype=torch.float64)] * (nproj // 2))
    elif kind == "column":  # one wide column and row, the rest diagonal
        dij = torch.diag(r.diagonal())
        dij[:, 5] = r[:, 5]
        dij[5] = r[:, 5]
    elif kind == "dense":
        dij = r
    dij = dij + dij.T
    say(f"D multiply, {kind} {dtype}")
    h, c, want = _case(nproj, dij, nb)
    h.set_flags(L.GW_PLAN_TIMING)
    got = h.apply(c.to(dev(), dtype)).cpu().to(torch.complex128)
    calls = h.stage_times()["dmul"][1]
    assert _rel(got, want) < tol
    assert calls == (1 if apart else 0)
