"""The Lanczos step kernels (csrc/krylov.hip) where they can go wrong: basis
lengths at the edges of the rows form (a single pair, one workgroup, one
element pair past it, odd lengths, the longest), every basis size up to a
restart, and the tridiagonal solver on spectra that its root prediction and
its twisted factorisation find hard.

Tolerances: an eigenpair stopped at residual 1e-12 |H| has its energy within
(1e-12)^2 / gap of exact, far below 1e-12 |H|; the tridiagonal solver brackets
the root to a few ulp of |T|, 1e-13 |T| with the reduction to tridiagonal form.
"""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import dmrg_ref as o

pytestmark = pytest.mark.gpu


def lib():
    from tnpy_amd import _lib

    return _lib.lib()


def stream():
    return torch.cuda.current_stream().cuda_stream


def symmetric_problem(rng, chil, d, chir, D=3):
    """Random environments with L[., w, .], R[., v, .] and W[w, v, ., .]
    symmetric matrices, so H_eff is symmetric."""
    def sym(n, k):
        a = rng.standard_normal((n, k, n))
        return a + a.transpose(2, 1, 0)

    W = rng.standard_normal((D, D, d, d))
    return sym(chil, D), W + W.transpose(0, 1, 3, 2), sym(chir, D)


@pytest.mark.parametrize("steps", [0, 1, 8])
@pytest.mark.parametrize("chil, d, chir, max_basis", [
    (1, 2, 1, 64), (1, 2, 2, 64), (3, 3, 3, 64), (8, 2, 8, 64), (5, 2, 13, 64), (8, 2, 9, 17), (16, 2, 31, 33),
    (24, 2, 24, 64), (33, 3, 5, 48), (12, 2, 11, 5)])
def test_lowest_pair(gpu, chil, d, chir, max_basis, steps):
    """steps 0: the single-problem solver; else the batched one, reading
    statuses every `steps` steps."""
    from tnpy_amd import _lib

    print(f"lowest pair {chil} {d} {chir} basis {max_basis} steps {steps}", flush=True)
    rng = np.random.default_rng(chil * 100 + chir)
    B = 1 if steps == 0 else 3
    probs = [symmetric_problem(rng, chil, d, chir) for _ in range(B)]
    N = chil * d * chir
    v0 = rng.standard_normal((B, N))
    L, W, R = (torch.from_numpy(np.stack([p[i] for p in probs])).cuda() for i in range(3))
    x = torch.from_numpy(v0).cuda()
    vec, hvec = torch.empty_like(x), torch.empty_like(x)
    opts = _lib.EigshOpts(tol=1e-12, max_basis=max_basis, max_matvecs=5000, precision=0, keep=0,
                          steps_per_check=max(steps, 1))
    infos = (_lib.EigshInfo * B)()
    args = [t.data_ptr() for t in (L, W, R, x, vec, hvec)] + [chil, 3, 3, d, chir]
    if steps == 0:
        ws = torch.empty(lib().tnx_eigsh_heff1_workspace_bytes(chil, 3, 3, d, chir, max_basis), dtype=torch.uint8,
                         device="cuda")
        st = lib().tnx_eigsh_heff1(*args, C.byref(opts), infos, ws.data_ptr(), ws.numel(), stream())
    else:
        ws = torch.empty(lib().tnx_eigsh_heff1_batched_workspace_bytes(chil, 3, 3, d, chir, max_basis, B),
                         dtype=torch.uint8, device="cuda")
        st = lib().tnx_eigsh_heff1_batched(*args, B, C.byref(opts), infos, ws.data_ptr(), ws.numel(), stream())
    assert st == 0
    for b, (Lh, Wh, Rh) in enumerate(probs):
        H = o.heff_dense(Lh, Wh, Rh)
        w = np.linalg.eigvalsh(H)
        nrm = np.abs(w).max()
        v, hv = vec[b].cpu().numpy(), hvec[b].cpu().numpy()
        assert infos[b].converged == 1
        assert abs(infos[b].eval - w[0]) <= 1e-12 * nrm
        assert abs(np.linalg.norm(v) - 1.0) < 1e-12
        assert np.linalg.norm(H @ v - infos[b].eval * v) <= 4e-12 * nrm
        assert np.linalg.norm(H @ v - hv) <= 1e-12 * nrm


@pytest.mark.parametrize("chi", [181, 256, 258])
def test_long_vectors(gpu, chi):
    """N = 65522 and 131072 (the rows form) and 133128 (the streaming one):
    the pair against the operator itself."""
    from tnpy_amd import _lib

    print(f"long vectors chi {chi}", flush=True)
    rng = np.random.default_rng(chi)
    L, W, R = (torch.from_numpy(a).cuda() for a in symmetric_problem(rng, chi, 2, chi))
    N = 2 * chi * chi
    x = torch.from_numpy(rng.standard_normal(N)).cuda()
    vec, hvec, hv = torch.empty_like(x), torch.empty_like(x), torch.empty_like(x)
    opts = _lib.EigshOpts(tol=1e-10, max_basis=64, max_matvecs=3000, precision=0, keep=20)
    info = _lib.EigshInfo()
    ws = torch.empty(lib().tnx_eigsh_heff1_workspace_bytes(chi, 3, 3, 2, chi, 64), dtype=torch.uint8, device="cuda")
    st = lib().tnx_eigsh_heff1(L.data_ptr(), W.data_ptr(), R.data_ptr(), x.data_ptr(), vec.data_ptr(),
                               hvec.data_ptr(), chi, 3, 3, 2, chi, C.byref(opts), C.byref(info), ws.data_ptr(),
                               ws.numel(), stream())
    assert st == 0 and info.converged == 1
    assert lib().tnx_heff1_matvec(L.data_ptr(), W.data_ptr(), R.data_ptr(), vec.data_ptr(), hv.data_ptr(), chi, 3, 3,
                                  2, chi, 0, ws.data_ptr(), ws.numel(), stream()) == 0
    assert abs(float(vec.norm()) - 1.0) < 1e-11
    assert float((hv - info.eval * vec).norm()) <= 2e-10 * info.anorm
    assert float((hv - hvec).norm()) <= 1e-11 * info.anorm


def spectra():
    rng = np.random.default_rng(5)
    Q = lambda n: np.linalg.qr(rng.standard_normal((n, n)))[0]  # noqa: E731
    yield "diagonal", np.diag(np.arange(40.0) - 7.0)
    yield "identity", np.eye(70)
    yield "zero", np.zeros((30, 30))
    a = 2.0 * np.eye(40) - np.eye(40, k=1) - np.eye(40, k=-1)
    a[19, 20] = a[20, 19] = 0.0
    yield "two equal blocks", a
    yield "laplacian", 2.0 * np.eye(130) - np.eye(130, k=1) - np.eye(130, k=-1)
    for n in (20, 100, 200):
        q = Q(n)
        yield f"cluster {n}", (q * np.concatenate([-5.0 + 1e-9 * np.arange(4), np.linspace(-4, 8, n - 4)])) @ q.T
        yield f"isolated {n}", (q * np.concatenate([[-1e6], rng.standard_normal(n - 1)])) @ q.T
        yield f"near zero {n}", (q * np.concatenate([[1e-12], np.linspace(1, 2, n - 1)])) @ q.T
        yield f"scaled down {n}", 1e-60 * (q * np.linspace(-1, 1, n)) @ q.T
        yield f"scaled up {n}", 1e60 * (q * np.linspace(-1, 1, n)) @ q.T


@pytest.mark.parametrize("name, M", list(spectra()), ids=[n for n, _ in spectra()])
def test_tridiagonal_solver(gpu, name, M):
    M = 0.5 * (M + M.T)
    n = M.shape[0]
    print(f"tridiagonal {name}", flush=True)
    md = torch.from_numpy(np.ascontiguousarray(M)).cuda()
    v = torch.empty(n, dtype=torch.float64, device="cuda")
    ev = C.c_double()
    ws = torch.empty(lib().tnx_syev_lowest_workspace_bytes(n), dtype=torch.uint8, device="cuda")
    assert lib().tnx_syev_lowest(md.data_ptr(), n, v.data_ptr(), C.byref(ev), ws.data_ptr(), ws.numel(),
                                 stream()) == 0
    w = np.linalg.eigvalsh(M)
    nrm = max(np.abs(w).max(), 1e-300)
    vh = v.cpu().numpy()
    assert abs(ev.value - w[0]) <= 1e-13 * nrm
    assert abs(np.linalg.norm(vh) - 1.0) < 1e-12
    assert np.linalg.norm((M / nrm) @ vh - (ev.value / nrm) * vh) <= 1e-12
