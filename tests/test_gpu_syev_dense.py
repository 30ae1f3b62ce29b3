"""Lowest eigenpair of dense matrices at the edges of the tridiagonalisation's
register layouts (32, 64, 128 and 192 rows), single and batched.

Tolerances: the tridiagonalisation is orthogonal, so eigenvalue and residual
carry its rounding, a small multiple of n eps of the norm (4 n eps here; the
eigenvector's norm that of its n-term sums)."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def api():
    from tnpy_amd import _lib

    return _lib


def matrix(kind, n, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((n, n))
    m = x + x.T
    if kind == "tridiagonal":  # every reflector is trivial
        m = np.triu(np.tril(m, 1), -1)
    elif kind == "blocks":  # reflectors vanish along the way
        m[: n // 2, n // 2:] = 0.0
        m[n // 2:, : n // 2] = 0.0
    elif kind == "scaled":
        m *= 1e-120
    return m


def check_pair(m, val, vec):
    w = np.linalg.eigvalsh(m)
    nrm = np.abs(w).max()
    assert abs(val - w[0]) <= 4 * len(m) * EPS * nrm
    assert abs(np.linalg.norm(vec) - 1.0) <= 4 * len(m) * EPS
    # the inverse iteration stops a little above the rounding of M v
    assert np.linalg.norm(m @ vec - val * vec) <= 16 * len(m) * EPS * nrm


@pytest.mark.parametrize("kind", ["full", "tridiagonal", "blocks", "scaled"])
@pytest.mark.parametrize("n", [2, 3, 5, 31, 32, 33, 63, 64, 65, 127, 128, 129, 162, 191, 192, 193, 256])
def test_lowest_pair(gpu, n, kind):
    print(f"syev {kind} {n}", flush=True)
    L = api().lib()
    m = matrix(kind, n, n)
    md = torch.from_numpy(m).cuda()
    vec, val = torch.empty(n, dtype=torch.float64, device="cuda"), C.c_double()
    nb = L.tnx_syev_lowest_workspace_bytes(n)
    buf = torch.empty(nb, dtype=torch.uint8, device="cuda")
    api().check(L.tnx_syev_lowest(md.data_ptr(), n, vec.data_ptr(), C.byref(val), buf.data_ptr(), nb,
                                  torch.cuda.current_stream().cuda_stream), "syev")
    check_pair(m, val.value, vec.cpu().numpy())
    assert np.array_equal(md.cpu().numpy(), m)


@pytest.mark.parametrize("n, batch", [(8, 5), (33, 3), (128, 4), (180, 2), (230, 2)])
def test_lowest_pair_batched(gpu, n, batch):
    print(f"syev batched {batch} x {n}", flush=True)
    L = api().lib()
    kinds = ["full", "blocks", "full", "tridiagonal", "full"][:batch]
    m = np.stack([matrix(k, n, 10 * n + i) for i, k in enumerate(kinds)])
    md = torch.from_numpy(m).cuda()
    vec, val = torch.empty(batch, n, dtype=torch.float64, device="cuda"), (C.c_double * batch)()
    nb = L.tnx_syev_lowest_batched_workspace_bytes(n, batch)
    buf = torch.empty(nb, dtype=torch.uint8, device="cuda")
    api().check(L.tnx_syev_lowest_batched(md.data_ptr(), n, batch, vec.data_ptr(), val, buf.data_ptr(), nb,
                                          torch.cuda.current_stream().cuda_stream), "syev_batched")
    for i in range(batch):
        check_pair(m[i], val[i], vec[i].cpu().numpy())
