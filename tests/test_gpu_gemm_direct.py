"""The register-operand GEMM of FP64 and FP32 (csrc/gemm_direct.h) at the
sizes where it can go wrong: tile edges, one index past a tile, odd extents,
partial groups of k, the K parts, small and many tiles, every layout and
operand type, bases and leading dimensions of any alignment, and operands
whose surroundings are NaN. Reference: numpy FP64 on the same values.

Tolerances (relative Frobenius): a sum of K products accumulated in FP64 is
within K * 1.1e-16 of exact, 6e-14 at the largest K here; in FP32 the
operands are rounded (6e-8) and K / 4 accumulations add sqrt(K / 4) * 6e-8,
1e-6 at the largest K.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {0: 6e-14, 1: 1e-6}


def lib():
    from tnpy_amd import _lib

    return _lib.lib()


def place(a, ld, off, f32):
    """`a` (rows x cols) in a NaN-filled device buffer with leading dimension
    ld, its first element `off` elements into the buffer; (buffer, address)."""
    rows, cols = a.shape
    dt = np.float32 if f32 else np.float64
    buf = np.full(off + rows * ld + 3, np.nan, dtype=dt)
    view = np.lib.stride_tricks.as_strided(buf[off:], (rows, cols), (ld * dt().itemsize, dt().itemsize))
    view[:] = a
    t = torch.from_numpy(buf).cuda()
    return t, t.data_ptr() + off * dt().itemsize


def run(M, N, K, ak, bn, prec, a32, b32, c32, pad, off, alpha, beta, seed):
    rng = np.random.default_rng(seed)
    A, B, C0 = rng.standard_normal((M, K)), rng.standard_normal((K, N)), rng.standard_normal((M, N))
    if a32:
        A = A.astype(np.float32).astype(np.float64)
    if b32:
        B = B.astype(np.float32).astype(np.float64)
    if c32:
        C0 = C0.astype(np.float32).astype(np.float64)
    lda, ldb, ldc = (K if ak else M) + pad, (N if bn else K) + pad, N + pad
    ta, pa = place(A if ak else A.T, lda, off, a32)
    tb, pb = place(B if bn else B.T, ldb, off, b32)
    tc, pc = place(C0, ldc, off, c32)
    st = lib().tnx_gemm(M, N, K, 1, alpha, pa, int(a32), lda, 0, ak, pb, int(b32), ldb, 0, bn, beta, pc, int(c32),
                        ldc, 0, prec, torch.cuda.current_stream().cuda_stream)
    assert st == 0
    torch.cuda.synchronize()
    out = tc.cpu().numpy().astype(np.float64)
    got = np.lib.stride_tricks.as_strided(out[off:], (M, N), (ldc * 8, 8)).copy()
    # nothing outside C is written: the padding is still NaN
    mask = np.ones(out.size, dtype=bool)
    for m in range(M):
        mask[off + m * ldc:off + m * ldc + N] = False
    assert np.isnan(out[mask]).all()
    want = alpha * A @ B + beta * C0
    assert np.linalg.norm(got - want) <= (TOL[prec] + (6e-8 if c32 else 0.0)) * np.linalg.norm(want)
    return got


SHAPES = [(1, 5, 3), (2, 2, 2), (2, 3, 1), (5, 1, 9), (16, 16, 8), (17, 17, 17), (16, 33, 7), (33, 16, 31),
          (65, 81, 40), (64, 129, 33), (128, 300, 64), (96, 96, 513), (31, 1000, 127), (300, 20, 64), (257, 641, 65)]


@pytest.mark.parametrize("ak, bn", [(1, 1), (1, 0), (0, 1), (0, 0)])
@pytest.mark.parametrize("M, N, K", SHAPES)
def test_edges(gpu, M, N, K, ak, bn):
    print(f"gemm direct {M}x{N}x{K} ak={ak} bn={bn}", flush=True)
    for prec in (0, 1):
        run(M, N, K, ak, bn, prec, 0, 0, 0, pad=3, off=1, alpha=0.75, beta=-0.5, seed=M + N + K)
        run(M, N, K, ak, bn, prec, 0, 0, 0, pad=0, off=0, alpha=1.0, beta=0.0, seed=M + N + K)


@pytest.mark.parametrize("a32, b32, c32", [(0, 1, 0), (0, 1, 1), (1, 0, 1), (1, 1, 0), (1, 1, 1)])
@pytest.mark.parametrize("M, N, K", [(17, 33, 9), (64, 160, 130), (520, 810, 40)])
def test_types(gpu, M, N, K, a32, b32, c32):
    print(f"gemm direct types {M}x{N}x{K} {a32}{b32}{c32}", flush=True)
    for prec in (0, 1):
        for ak, bn in ((1, 1), (0, 1), (1, 0)):
            run(M, N, K, ak, bn, prec, a32, b32, c32, pad=1, off=1, alpha=1.0, beta=0.5, seed=7)


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("M, N, K", [(1000, 2000, 96), (2048, 2560, 72), (700, 900, 640), (400, 1200, 100)])
def test_large_tiles(gpu, prec, M, N, K):
    """Shapes whose rule picks the wide wave tiles and the K parts."""
    print(f"gemm direct large {M}x{N}x{K}", flush=True)
    for ak, bn in ((1, 1), (0, 1), (1, 0)):
        for f in (0, 1):
            run(M, N, K, ak, bn, prec, f and prec, f and prec, 0, pad=0, off=0, alpha=1.0, beta=1.0, seed=3)


def test_alignment_same_bits(gpu):
    """Base alignment and leading dimension change no bit."""
    ref = run(130, 181, 93, 1, 1, 0, 0, 0, 0, pad=0, off=0, alpha=1.0, beta=0.0, seed=1)
    for pad, off in ((1, 0), (0, 1), (5, 3)):
        assert np.array_equal(run(130, 181, 93, 1, 1, 0, 0, 0, 0, pad=pad, off=off, alpha=1.0, beta=0.0, seed=1), ref)


def test_non_finite_stay_in_their_rows(gpu):
    """An infinity and a NaN reach the rows and columns they belong to only,
    partial tiles and K tails included."""
    rng = np.random.default_rng(0)
    M, N, K = 37, 41, 21
    A, B = rng.standard_normal((M, K)), rng.standard_normal((K, N))
    A[36, 20] = np.inf
    B[3, 40] = np.nan
    Ad, Bd = torch.from_numpy(A).cuda(), torch.from_numpy(B).cuda()
    C = torch.zeros(M, N, dtype=torch.float64, device="cuda")
    assert lib().tnx_gemm_f64(M, N, K, 1, 1.0, Ad.data_ptr(), K, 0, 1, Bd.data_ptr(), N, 0, 1, 0.0, C.data_ptr(), N,
                              0, 0, torch.cuda.current_stream().cuda_stream) == 0
    got = C.cpu().numpy()
    assert np.isfinite(got[:36, :40]).all()
    assert np.isnan(got[:, 40]).all() and np.isinf(got[36, :40]).all()
