"""The generalized Davidson solver's matrix-vector products over its basis run
on many workgroups: each is one output tile with K = chi d chi.

The limit: a step reads up to 24 basis rows about eight times, 50 MB at chi =
128, 0.6 ms at a hundredth of the memory's rate; some 40 launches of 20 us and
2 ms for the projected problem come to 3.4 ms together, 5 are allowed. With
each product on one workgroup a step takes 16."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_step_time(gpu):
    from tnpy_amd import _lib

    print("generalized eigensolver step time", flush=True)
    L = _lib.lib()
    chi, D, d, basis = 128, 3, 2, 24
    N = chi * d * chi
    rng = np.random.default_rng(1)

    def sym(k):
        a = rng.standard_normal((chi, k, chi))
        return torch.from_numpy(a + a.transpose(2, 1, 0)).cuda()

    W = rng.standard_normal((D, D, d, d))
    Le, We, Re = sym(D), torch.from_numpy(W + W.transpose(0, 1, 3, 2)).cuda(), sym(D)
    # M_eff = 1
    eye = torch.eye(chi, dtype=torch.float64, device="cuda").reshape(chi, 1, chi).contiguous()
    W2 = torch.eye(d, dtype=torch.float64, device="cuda").reshape(1, 1, d, d).contiguous()
    x = torch.from_numpy(rng.standard_normal(N)).cuda()
    vec, hvec = torch.empty_like(x), torch.empty_like(x)
    opts = _lib.EigshOpts(tol=1e-13, max_basis=basis, max_matvecs=80, precision=0, keep=8)
    info = _lib.EigshInfo()
    nb = L.tnx_eigsh_gen_heff1_workspace_bytes(chi, D, D, 1, 1, d, chi, basis)
    ws = torch.empty(nb, dtype=torch.uint8, device="cuda")

    def solve():
        st = L.tnx_eigsh_gen_heff1(Le.data_ptr(), We.data_ptr(), Re.data_ptr(), eye.data_ptr(), W2.data_ptr(),
                                   eye.data_ptr(), x.data_ptr(), vec.data_ptr(), hvec.data_ptr(), chi, D, D, 1, 1, d,
                                   chi, C.byref(opts), C.byref(info), ws.data_ptr(), nb,
                                   torch.cuda.current_stream().cuda_stream)
        assert st in (_lib.TNX_OK, _lib.TNX_ERR_NOCONV)

    solve()
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    a.record()
    solve()
    b.record()
    b.synchronize()
    assert info.matvecs >= 40  # two a step
    assert a.elapsed_time(b) / (info.matvecs / 2) <= 5.0
