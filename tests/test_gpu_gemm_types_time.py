"""FP64 products with an FP32 left operand run the same kernel as FP64 ones: it
reads fewer bytes and adds a conversion per loaded value, so half as long again
is the limit (the LDS-tile kernel takes 2.8 times as long)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_float_left_operand(gpu):
    from tnpy_amd import _lib

    print("FP64 gemm with a float left operand", flush=True)
    L = _lib.lib()
    M, N, K = 1024, 2048, 2048
    B = torch.randn(K, N, dtype=torch.float64, device="cuda")
    out = torch.empty(M, N, dtype=torch.float64, device="cuda")

    def time(dt):
        A = torch.randn(M, K, dtype=dt, device="cuda")
        best = 1e9
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            st = L.tnx_gemm(M, N, K, 1, 1.0, A.data_ptr(), int(dt == torch.float32), K, 0, 1, B.data_ptr(), 0, N, 0, 1,
                            0.0, out.data_ptr(), 0, N, 0, 0, torch.cuda.current_stream().cuda_stream)
            b.record()
            b.synchronize()
            assert st == 0
            best = min(best, a.elapsed_time(b))
        return best

    assert time(torch.float32) <= 1.5 * time(torch.float64)
