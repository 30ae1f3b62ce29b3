"""Lowest eigenpair where the lowest level is degenerate, exactly (the
tridiagonal form falls apart and its blocks share the level) or to rounding.

Tolerances: reduction to tridiagonal form and back are n reflectors of a few
eps |M| each, the tridiagonal pair has a residual of 6 eps times its row-sum
norm (at most 3 |M|): (8 n + 18) eps |M| together, below 16 n eps |M| for n >=
3 (n = 2 needs no reflectors: 18 eps). The energy is within the residual."""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def api():
    from tnpy_amd import _lib

    return _lib


def chain(n, xy, z):
    """sum_i xy (S+S- + S-S+) / 2 + z SzSz over an open chain."""
    sp, sz = np.array([[0.0, 1.0], [0.0, 0.0]]), np.diag([0.5, -0.5])
    H = np.zeros((2**n, 2**n))
    for i in range(n - 1):
        two = xy * 0.5 * (np.kron(sp, sp.T) + np.kron(sp.T, sp)) + z * np.kron(sz, sz)
        H += np.kron(np.kron(np.eye(2**i), two), np.eye(2 ** (n - i - 2)))
    return H


def blocks(*bs):
    n = sum(len(b) for b in bs)
    out, at = np.zeros((n, n)), 0
    for b in bs:
        out[at:at + len(b), at:at + len(b)] = b
        at += len(b)
    return out


def exact_cases():
    x = np.array([[0.0, 1.0], [1.0, 0.0]])
    yield "1 0 0", np.diag([1.0, 0.0, 0.0])
    yield "1 -1 -1 1", np.diag([1.0, -1.0, -1.0, 1.0])
    yield "3 -2 -2 5", np.diag([3.0, -2.0, -2.0, 5.0])
    yield "two swaps", blocks(x, x)
    yield "swaps apart", blocks(np.diag([2.0]), x, np.diag([0.5]), x, np.diag([3.0]))
    yield "far scale", 1e-70 * np.diag([3.0, -2.0, -2.0, 5.0])
    yield "70 rows", np.diag(np.where(np.arange(70) % 23 == 11, -3.0, 1.0))
    yield "200 rows", np.diag(np.where(np.arange(200) % 67 == 66, -3.0, np.arange(200.0)))
    for n in range(2, 8):
        yield f"ising {n}", chain(n, 0.0, 1.0)
    yield "heisenberg 3", chain(3, 1.0, 1.0)


def check_pair(m, val, vec):
    n = len(m)
    w = np.linalg.eigvalsh(m)
    nrm = np.abs(w).max()
    tol = 16 * max(n, 3) * EPS
    assert abs(val - w[0]) <= tol * nrm
    assert abs(np.linalg.norm(vec) - 1.0) <= tol
    assert np.linalg.norm(m @ vec - val * vec) <= tol * nrm


def lowest(ms):
    """Single (one matrix) or batched."""
    L, batch, n = api().lib(), len(ms), ms.shape[1]
    stream = torch.cuda.current_stream().cuda_stream
    md = torch.from_numpy(np.ascontiguousarray(ms)).cuda()
    vec, val = torch.empty(batch, n, dtype=torch.float64, device="cuda"), (C.c_double * batch)()
    nb = L.tnx_syev_lowest_workspace_bytes(n) if batch == 1 else L.tnx_syev_lowest_batched_workspace_bytes(n, batch)
    buf = torch.empty(nb, dtype=torch.uint8, device="cuda")
    if batch == 1:
        api().check(L.tnx_syev_lowest(md.data_ptr(), n, vec.data_ptr(), val, buf.data_ptr(), nb, stream), "syev")
    else:
        api().check(L.tnx_syev_lowest_batched(md.data_ptr(), n, batch, vec.data_ptr(), val, buf.data_ptr(), nb,
                                              stream), "syev_batched")
    return np.array(val), vec.cpu().numpy()


@pytest.mark.parametrize("name, m", list(exact_cases()), ids=[n for n, _ in exact_cases()])
def test_exactly_degenerate(gpu, name, m):
    print(f"degenerate {name}", flush=True)
    val, vec = lowest(m[None])
    check_pair(m, val[0], vec[0])
    val, vec = lowest(np.stack([m, -m, m]))
    for i, mi in enumerate([m, -m, m]):
        check_pair(mi, val[i], vec[i])


@pytest.mark.parametrize("sites, count", [(3, 300), (5, 300), (7, 20)])
def test_degenerate_to_rounding(gpu, sites, count):
    """An odd Heisenberg chain (a doublet below) in random bases."""
    print(f"rotated heisenberg {sites}", flush=True)
    rng = np.random.default_rng(sites)
    H = chain(sites, 1.0, 1.0)
    ms = []
    for _ in range(count):
        q = np.linalg.qr(rng.standard_normal(H.shape))[0]
        m = q @ H @ q.T
        ms.append(0.5 * (m + m.T))
    ms = np.stack(ms)
    val, vec = lowest(ms)
    for m, v, x in zip(ms, val, vec):
        check_pair(m, v, x)


def test_two_site_ising_chain(gpu):
    """A two-site chain of SzSz only from a product state: the local H_eff is
    diagonal with a degenerate lowest level, -1/4."""
    from tnpy_amd import FiniteDMRG, MatrixProductOperator, MatrixProductState

    print("two-site ising chain", flush=True)
    sz = np.diag([0.5, -0.5])
    mpo = MatrixProductOperator([sz[None], sz[None]])
    eye = np.eye(2)
    mps = MatrixProductState([eye.reshape(1, 2, 2) / np.sqrt(2.0), eye.reshape(2, 2, 1)])
    dmrg = FiniteDMRG(mpo=mpo, bond_dim=2, mps=mps)
    for site in range(2):
        energy, psi = dmrg.one_site_solver(site)
        H = dmrg.environment.one_site_full_matrix(site)
        x = np.asarray(psi).ravel()
        assert abs(energy - np.linalg.eigvalsh(H)[0]) <= 48 * EPS
        assert np.linalg.norm(H @ x - energy * x) <= 48 * EPS * np.linalg.norm(x)
