"""Truncated SVD and dense eigenproblems whose core is one block pair (at most
64 rows, all Jacobi sweeps in one launch) and just past it.

Tolerances: rows are orthogonal to 1e-14 of their norms, so singular values
are within n eps of s_max; U comes from a QR of the normalised rows."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def matrix(kind, a, b):
    rng = np.random.default_rng(100 * a + b)
    x = rng.standard_normal((a, b))
    n = min(a, b)
    if kind == "graded":
        u, v = np.linalg.qr(rng.standard_normal((a, n)))[0], np.linalg.qr(rng.standard_normal((b, n)))[0]
        x = (u * np.logspace(0, -18, n)) @ v.T
    elif kind == "rank":
        r = max(1, n // 3)
        x = rng.standard_normal((a, r)) @ rng.standard_normal((r, b))
    elif kind == "zero":
        x[:] = 0.0
    elif kind == "tiny":
        x *= 1e-60
    return x


@pytest.mark.parametrize("kind", ["random", "graded", "rank", "zero", "tiny"])
@pytest.mark.parametrize("a, b", [(1, 1), (2, 3), (31, 32), (33, 32), (64, 64), (128, 63), (40, 200), (65, 65), (66, 90)])
def test_singular_triplets(gpu, a, b, kind):
    from tnpy_amd import _lib

    print(f"svd {kind} {a}x{b}", flush=True)
    x = matrix(kind, a, b)
    n = min(a, b)
    for k in sorted({1, (n + 1) // 2, n}):
        u, y, sv = _lib.svd_trunc(torch.from_numpy(x).cuda(), k)
        u, y = u.cpu().numpy(), y.cpu().numpy()
        s = np.linalg.svd(x, compute_uv=False)
        assert np.abs(sv - s[:k]).max() <= 16 * (a + b) * EPS * s[0]
        assert np.abs(u.T @ u - np.eye(k)).max() <= EPS * (a + 20 * n)
        assert np.abs(y - u.T @ x).max() <= 16 * (a + b) * EPS * s[0]
        if kind in ("random", "rank"):
            # the discarded weight is the least possible one
            rest = np.sqrt(np.sum(s[k:] ** 2))
            assert abs(np.linalg.norm(x - u @ y) - rest) <= 1e-7 * rest + 16 * (a + b) * EPS * s[0]
