"""Cholesky QR with regularised pivots: matrices that fit in LDS (one
workgroup), its transposed and batched forms, and larger matrices in wide
panels; Householder where squares leave the range of the numbers.

Tolerances: Q is formed by one triangular solve from columns orthonormal to
0.1, so |Q^T Q - I| carries the rounding of m-term and n-term sums, eps (m +
10 n); every column of A - Q R carries the rounding of n-term sums per pass,
10 n eps of the column's norm."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps

# edges of the 16-wide tiles, of the two LDS sizes and of the largest shapes
SHAPES = [(1, 1), (2, 1), (16, 16), (17, 16), (33, 17), (64, 32), (65, 33), (96, 48), (48, 48), (120, 60), (128, 64),
          (144, 72), (80, 80), (1000, 16), (300, 48)]
# past the LDS limit: one panel, edges of a second and a third, long and square
WIDE = [(160, 80), (128, 128), (129, 129), (500, 100), (257, 131), (259, 259), (520, 257), (600, 300), (401, 399),
        (5000, 17), (8192, 33), (1200, 640)]


def matrix(kind, m, n):
    rng = np.random.default_rng(1000 * m + n)
    a = rng.standard_normal((m, n))
    if kind == "graded":  # singular values over 16 decades
        u, v = np.linalg.qr(a)[0], np.linalg.qr(rng.standard_normal((n, n)))[0]
        a = (u * np.logspace(0, -16, n)) @ v.T
    elif kind == "rank":
        r = max(1, n // 5)
        a = rng.standard_normal((m, r)) @ rng.standard_normal((r, n))
    elif kind == "equal":
        a[:, n // 2] = a[:, 0]
        a[:, -1] = a[:, 0]
    elif kind == "zero":
        a[:, n // 3] = 0.0
        a[:, n // 2:n // 2 + 3] = 0.0
    elif kind == "null":
        a[:] = 0.0
    elif kind in ("huge", "tiny"):  # squares past 1e290 and below 1e-290
        a *= 1e147 if kind == "huge" else 1e-147
    elif kind == "scaled":  # columns over 200 decades
        a *= 10.0 ** rng.uniform(-100, 100, n)
    return a


def check_qr(a, q, r):
    m, n = a.shape
    assert np.all(np.tril(r, -1) == 0.0) and np.all(np.diag(r) >= 0.0)
    assert np.abs(q.T @ q - np.eye(n)).max() <= EPS * (m + 10 * n)
    scale = np.linalg.norm(a / np.maximum(np.abs(a).max(axis=0), 1e-300), axis=0) * np.abs(a).max(axis=0)
    assert np.all(np.linalg.norm((a - q @ r) / np.maximum(scale, 1e-300), axis=0) <= 10 * n * EPS)


def lib():
    from tnpy_amd import _lib

    return _lib


def workspace(nbytes):
    buf = torch.empty(max(1, nbytes), dtype=torch.uint8, device="cuda")
    return buf, buf.data_ptr(), nbytes


@pytest.mark.parametrize("kind", ["random", "graded", "rank", "equal", "zero", "null", "scaled", "huge", "tiny"])
@pytest.mark.parametrize("m, n", SHAPES + WIDE)
def test_qr(gpu, m, n, kind):
    print(f"qr {kind} {m}x{n}", flush=True)
    L = lib().lib()
    a = matrix(kind, m, n)
    ad, r = torch.from_numpy(a.copy()).cuda(), torch.full((n, n), 7.0, dtype=torch.float64, device="cuda")
    buf, wp, wb = workspace(L.tnx_qr_workspace_bytes(m, n))
    lib().check(L.tnx_qr(ad.data_ptr(), m, n, r.data_ptr(), wp, wb, torch.cuda.current_stream().cuda_stream), "qr")
    q, r = ad.cpu().numpy(), r.cpu().numpy()
    check_qr(a, q, r)
    if kind == "random":
        # the factorisation with a non-negative diagonal is unique
        q0, r0 = np.linalg.qr(a)
        s = np.where(np.diag(r0) < 0, -1.0, 1.0)
        cond = np.linalg.cond(a)
        assert np.abs(q - q0 * s).max() <= 100 * n * EPS * cond


@pytest.mark.parametrize("chi", [7, 24, 60])
def test_gauge_left_in_lds(gpu, chi):
    """The transposed form, and a batch in which one matrix takes the
    Householder steps (huge): each the same as its matrix alone."""
    L = lib().lib()
    st = torch.cuda.current_stream().cuda_stream
    kinds = ["random", "zero", "rank", "graded", "huge", "random"]
    a = np.stack([matrix(k, 2 * chi, chi).T.reshape(chi, 2, chi) * (1 + i) for i, k in enumerate(kinds)])
    prev = np.random.default_rng(chi).standard_normal((len(kinds), 5, chi))
    ad, pd = torch.from_numpy(a.copy()).cuda(), torch.from_numpy(prev).cuda()
    out = torch.empty_like(pd)
    buf, wp, wb = workspace(L.tnx_gauge_batched_workspace_bytes(chi, 2, chi, len(kinds)))
    lib().check(L.tnx_gauge_left_batched(ad.data_ptr(), pd.data_ptr(), out.data_ptr(), chi, 2, chi, 5, len(kinds),
                                         wp, wb, st), "gauge_left_batched")
    buf1, wp1, wb1 = workspace(L.tnx_gauge_workspace_bytes(chi, 2, chi))
    for i in range(len(kinds)):
        q = ad[i].cpu().numpy().reshape(chi, 2 * chi)
        assert np.abs(q @ q.T - np.eye(chi)).max() <= EPS * 12 * chi
        want = prev[i] @ a[i].reshape(chi, -1)
        assert np.linalg.norm(out[i].cpu().numpy() @ q - want) <= 20 * chi * EPS * np.linalg.norm(
            prev[i]) * np.linalg.norm(a[i])
        a1, o1 = torch.from_numpy(a[i].copy()).cuda(), torch.empty_like(pd[i])
        lib().check(L.tnx_gauge_left(a1.data_ptr(), pd[i].data_ptr(), o1.data_ptr(), chi, 2, chi, 5, wp1, wb1, st),
                    "gauge_left")
        assert torch.equal(a1, ad[i])
