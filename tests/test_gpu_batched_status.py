"""Batched Lanczos that reads the statuses after every step: the problems of a
large batch finish at different steps, and what the next step, queued for all
of them, left behind is finished for those that remain. The workspace is full
of NaN before the call.

Tolerances: a pair stopped at residual tol |H| has its energy within tol |H|
of an eigenvalue, and both solvers stop at the lowest one here (they start
from it, disturbed); the residual is recomputed with a matvec of 1e-14 |H|."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def api():
    from tnpy_amd import _lib

    return _lib


@pytest.mark.parametrize("chi, batch", [(36, 100), (64, 64)])
def test_problems_that_leave(gpu, chi, batch):
    print(f"batched statuses chi {chi} batch {batch}", flush=True)
    L = api().lib()
    stream = torch.cuda.current_stream().cuda_stream
    D, d, tol = 3, 2, 1e-9
    N = chi * d * chi
    g = torch.Generator().manual_seed(chi)

    def symmetric():
        a = torch.randn(batch, chi, D, chi, dtype=torch.float64, generator=g).cuda()
        return a + a.transpose(1, 3)

    Le, Re = symmetric().contiguous(), symmetric().contiguous()
    W = torch.randn(batch, D, D, d, d, dtype=torch.float64, generator=g).cuda()
    W = (W + W.transpose(3, 4)).contiguous()
    x = torch.randn(batch, N, dtype=torch.float64, generator=g).cuda()
    noise = torch.randn(batch, N, dtype=torch.float64, generator=g).cuda()
    nb = L.tnx_eigsh_heff1_batched_workspace_bytes(chi, D, D, d, chi, 64, batch)
    ws = torch.empty(nb // 8 + 1, dtype=torch.float64, device="cuda")

    def solve(start, steps):
        ws.fill_(float("nan"))
        vec, hvec = torch.empty_like(start), torch.empty_like(start)
        opts = api().EigshOpts(tol=tol, max_basis=64, max_matvecs=1500, precision=0, keep=0, steps_per_check=steps)
        info = (api().EigshInfo * batch)()
        api().check(L.tnx_eigsh_heff1_batched(Le.data_ptr(), W.data_ptr(), Re.data_ptr(), start.data_ptr(),
                                              vec.data_ptr(), hvec.data_ptr(), chi, D, D, d, chi, batch,
                                              C.byref(opts), info, ws.data_ptr(), ws.numel() * 8, stream), "eigsh")
        return vec, info

    ref, want = solve(x, 8)
    size = torch.tensor([10.0 ** -(1 + b % 8) for b in range(batch)], dtype=torch.float64, device="cuda")
    start = ref + size[:, None] * noise / noise.norm(dim=1, keepdim=True)
    vec, got = solve(start.contiguous(), 1)
    assert len({got[b].matvecs for b in range(batch)}) > 4  # they did leave at different steps
    hv = torch.empty_like(vec)
    api().check(L.tnx_heff1_matvec_batched(Le.data_ptr(), W.data_ptr(), Re.data_ptr(), vec.data_ptr(), hv.data_ptr(),
                                           chi, D, D, d, chi, batch, 0, ws.data_ptr(), ws.numel() * 8, stream), "mv")
    for b in range(batch):
        nrm = want[b].anorm
        assert got[b].converged == 1
        assert abs(got[b].eval - want[b].eval) <= 2 * tol * nrm
        assert abs(float(vec[b].norm()) - 1.0) <= 1e-12
        assert float((hv[b] - got[b].eval * vec[b]).norm()) <= 2 * tol * nrm
