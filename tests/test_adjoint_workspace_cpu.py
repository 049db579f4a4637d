"""Workspaces of the adjoint and eigensolver entry points, with a stand-in for the
library that records the pointers it is given: calls that overlap (two streams) get
memory of their own, and one call's memory is bounded."""

from types import SimpleNamespace

import pytest
import torch

from gradwave_amd import _lib as L
from gradwave_amd import adjoint as A


class _Library:
    """gw_hpsi_adjoint_v and gw_proj_phase_grad, recording (workspace, bytes); ``during``
    runs inside the first call, as another stream's call would."""

    def __init__(self, bytes_of, during=None):
        self.bytes_of, self.during, self.calls = bytes_of, during, []

    def gw_plan_info(self, handle, prec, info, n):
        info[2] = 2
        return 0

    def gw_hpsi_adjoint_v_workspace_bytes(self, handle, nb, prec):
        return self.bytes_of(nb)

    def gw_proj_phase_grad_workspace_bytes(self, nk, nproj):
        return self.bytes_of(nproj)

    def _call(self, **kw):
        self.calls.append(SimpleNamespace(**kw))
        if self.during is not None and len(self.calls) == 1:
            self.during()
        return 0

    def gw_hpsi_adjoint_v(self, handle, prec, c, ldc, sc, g, ldg, sg, nb, gv, ws, nbytes, stream):
        return self._call(c=c, g=g, nb=nb, ws=ws, bytes=nbytes)

    def gw_proj_phase_grad(self, nk, nproj, npw, na, gp, p, kpg, ai, gtau, ws, nbytes, stream):
        return self._call(ws=ws, bytes=nbytes)


@pytest.fixture
def install(monkeypatch):
    def put(lib):
        monkeypatch.setattr(L, "lib", lambda: lib)
        monkeypatch.setattr(L, "stream_ptr", lambda device=None: 0)
        return lib
    return put


def _block(nb):
    return torch.zeros(2, nb, 7, dtype=torch.complex128)


def _disjoint(a, b):
    return a.ws + a.bytes <= b.ws or b.ws + b.bytes <= a.ws


def test_overlapping_v_adjoints_do_not_share_a_workspace(install):
    op = SimpleNamespace(fwd=SimpleNamespace(plan=SimpleNamespace(handle=None)), shape=(4, 4, 4))
    lib = install(_Library(lambda nb: 4096 * nb, lambda: A.adjoint_v(op, _block(2), _block(2))))
    A.adjoint_v(op, _block(3), _block(3))
    assert len(lib.calls) == 2 and _disjoint(*lib.calls)


def test_overlapping_phase_adjoints_do_not_share_a_workspace(install):
    p = torch.zeros(2, 3, 7, dtype=torch.complex128)
    ctx = SimpleNamespace(saved_tensors=(p, torch.zeros(2, 7, 3), torch.zeros(3, dtype=torch.int64)), na=1)
    lib = install(_Library(lambda n: 4096 * n, lambda: A._ProjPhaseFn.backward(ctx, p)))
    A._ProjPhaseFn.backward(ctx, p)
    assert len(lib.calls) == 2 and _disjoint(*lib.calls)


def test_v_adjoint_goes_in_band_chunks_under_the_budget(install, monkeypatch):
    from gradwave_amd import hamiltonian

    monkeypatch.setattr(hamiltonian, "_LIB_FFT_BUDGET_BYTES", 3500)
    op = SimpleNamespace(fwd=SimpleNamespace(plan=SimpleNamespace(handle=None)), shape=(4, 4, 4))
    # one band is above the budget, three bands fit, a partial per group of two bands
    for per_band, group, chunks in ((9000, 0, [1] * 8), (1000, 0, [3, 3, 2]), (1000, 600, [2, 2, 2, 2]), (10, 0, [8])):
        lib = install(_Library(lambda nb: per_band * nb + group * ((nb + 1) // 2)))
        c, g = _block(8), _block(8)
        A.adjoint_v(op, c, g)
        assert [x.nb for x in lib.calls] == chunks
        done = 0
        for x in lib.calls:
            assert x.c == c.data_ptr() + done * c.stride(1) * 16 and x.g == g.data_ptr() + done * g.stride(1) * 16
            assert x.bytes >= lib.bytes_of(x.nb) and x.bytes <= max(3500, lib.bytes_of(1))
            done += x.nb


def test_overlapping_eigensolves_do_not_share_a_workspace(monkeypatch):
    from gradwave_amd import linalg as LA

    jobs = []

    class Lib:
        def gw_heev_workspace_bytes(self, n, nev):
            return 4096 * n

        def gw_heev_max_n(self):
            return 512

        def gw_heev_batched(self, count, arr, stream):
            jobs.append([(arr[i].ws, 4096 * arr[i].n) for i in range(count)])
            if len(jobs) == 1:  # another stream's call
                LA.eigh_lowest([torch.zeros(2, 3, 3, dtype=torch.complex128)], [1])
            return 0

    monkeypatch.setattr(L, "lib", lambda: Lib())
    monkeypatch.setattr(L, "stream_ptr", lambda device=None: 0)
    monkeypatch.setattr(L, "require_gpu", lambda t, name: None)
    LA.eigh_lowest([torch.zeros(3, 5, 5, dtype=torch.complex128)], [2])
    spans = sorted(jobs[0] + jobs[1])
    assert len(spans) == 5 and all(a[0] + a[1] <= b[0] for a, b in zip(spans, spans[1:]))
