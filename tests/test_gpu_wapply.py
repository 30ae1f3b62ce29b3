"""The W-apply kernel (csrc/contract.hip) through the contractions that use
it, at the row counts where its register form or its row tiles change (D d =
10, 12, 16, 24, 32, 50, 64 inputs and outputs, unequal ones), odd and
smallest inner bonds, and FP32 intermediates, against the oracle.

Tolerance: three chained sums of at most D d + 2 chi products each, FP64:
1e-13 relative (Frobenius); FP32 intermediates: 3e-5.
"""
import numpy as np
import pytest
import torch

from oracle import dmrg_ref as o

pytestmark = pytest.mark.gpu

SHAPES = [(3, 5, 5, 2, 1), (1, 5, 5, 2, 3), (7, 6, 6, 2, 9), (5, 8, 8, 2, 6), (4, 12, 10, 2, 5), (6, 16, 16, 2, 7),
          (9, 25, 25, 2, 11), (3, 32, 32, 2, 4), (4, 1, 32, 2, 6), (6, 32, 1, 2, 3), (5, 9, 9, 3, 5), (40, 5, 5, 2, 33)]


def relerr(a, b):
    return np.linalg.norm(a - b) / np.linalg.norm(b)


@pytest.mark.parametrize("prec, tol", [(0, 1e-13), (1, 3e-5)])
@pytest.mark.parametrize("shape", SHAPES)
def test_contractions(gpu, shape, prec, tol):
    from tnpy_amd import _lib

    lib = _lib.lib()
    chil, Dl, Dr, d, chir = shape
    print(f"W-apply {shape} prec {prec}", flush=True)
    rng = np.random.default_rng(sum(shape))
    L, R = rng.standard_normal((chil, Dl, chil)), rng.standard_normal((chir, Dr, chir))
    W, x = rng.standard_normal((Dl, Dr, d, d)), rng.standard_normal((chil, d, chir))
    Ld, Rd, Wd, xd = (torch.from_numpy(a).cuda() for a in (L, R, W, x))
    s = torch.cuda.current_stream().cuda_stream
    nb = max(lib.tnx_heff1_workspace_bytes(*shape), lib.tnx_env_workspace_bytes(*shape))
    ws = torch.empty(int(nb), dtype=torch.uint8, device="cuda")
    y = torch.empty_like(xd)
    assert lib.tnx_heff1_matvec(Ld.data_ptr(), Wd.data_ptr(), Rd.data_ptr(), xd.data_ptr(), y.data_ptr(), *shape,
                                prec, ws.data_ptr(), ws.numel(), s) == 0
    assert relerr(y.cpu().numpy().ravel(), o.heff_matvec(L, W, R, x).ravel()) < tol
    out = torch.empty(chir, Dr, chir, dtype=torch.float64, device="cuda")
    assert lib.tnx_env_left(Ld.data_ptr(), xd.data_ptr(), Wd.data_ptr(), out.data_ptr(), *shape, prec, ws.data_ptr(),
                            ws.numel(), s) == 0
    assert relerr(out.cpu().numpy(), o.env_left(L, x, W)) < tol
    out = torch.empty(chil, Dl, chil, dtype=torch.float64, device="cuda")
    assert lib.tnx_env_right(Rd.data_ptr(), xd.data_ptr(), Wd.data_ptr(), out.data_ptr(), *shape, prec, ws.data_ptr(),
                             ws.numel(), s) == 0
    assert relerr(out.cpu().numpy(), o.env_right(R, x, W)) < tol
