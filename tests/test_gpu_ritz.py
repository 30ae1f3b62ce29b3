"""Restarts of the Lanczos solver on clustered spectra: the projected matrix's
eigenvectors by twisted factorisations and, where clusters are too tight for
them, by implicit QL.

Tolerances: the solve stops at a residual of 1e-11 |H|, |H| its own estimate
(the norm of the projected matrix by rows); its energy is then
within 1e-11 |H| of an eigenvalue, and the lowest cluster is narrower than that
or resolved."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batched", [False, True])
@pytest.mark.parametrize("split", [1e-2, 1e-5, 1e-8, 1e-10, 1e-13, 0.0])
@pytest.mark.parametrize("max_basis", [24, 33, 64])
def test_clustered(gpu, max_basis, split, batched):
    from tnpy_amd import _lib

    print(f"clustered split {split} basis {max_basis} batched {batched}", flush=True)
    lib = _lib.lib()
    rng = np.random.default_rng(max_basis)
    chil, d, chir = 8, 2, 40
    # H = left x site x right: every product of a site and a right eigenvalue
    # is a cluster of 8, `split` wide
    left = np.diag(1.0 + split * rng.uniform(0, 1, chil))
    q = np.linalg.qr(rng.standard_normal((chir, chir)))[0]
    right = (q * np.sort(rng.uniform(-1.0, 0.5, chir))) @ q.T
    right = 0.5 * (right + right.T)
    site = np.diag([1.0, 0.7])
    h = np.kron(np.kron(left, site), right)
    n = len(h)
    w = np.linalg.eigvalsh(h)
    B = 2
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(np.stack([a] * B))).cuda()  # noqa: E731
    L, W, R = dev(left[:, None, :]), dev(site[None, None]), dev(right[:, None, :])
    x = torch.from_numpy(rng.standard_normal((B, n))).cuda()
    vec, hvec = torch.empty_like(x), torch.empty_like(x)
    opts = _lib.EigshOpts(tol=1e-11, max_basis=max_basis, max_matvecs=6000, precision=0, keep=0, steps_per_check=8)
    infos = (_lib.EigshInfo * B)()
    args = [t.data_ptr() for t in (L, W, R, x, vec, hvec)] + [chil, 1, 1, d, chir]
    st = torch.cuda.current_stream().cuda_stream
    if batched:
        nb = lib.tnx_eigsh_heff1_batched_workspace_bytes(chil, 1, 1, d, chir, max_basis, B)
        ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
        assert lib.tnx_eigsh_heff1_batched(*args, B, C.byref(opts), infos, ws.data_ptr(), nb, st) == 0
    else:
        nb = lib.tnx_eigsh_heff1_workspace_bytes(chil, 1, 1, d, chir, max_basis)
        ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
        assert lib.tnx_eigsh_heff1(*args, C.byref(opts), infos, ws.data_ptr(), nb, st) == 0
    for b in range(B if batched else 1):
        v = vec[b].cpu().numpy()
        assert infos[b].converged == 1
        assert abs(infos[b].eval - w[0]) <= 1e-11 * infos[b].anorm
        assert abs(np.linalg.norm(v) - 1.0) < 1e-12
        assert np.linalg.norm(h @ v - infos[b].eval * v) <= 4e-11 * infos[b].anorm
