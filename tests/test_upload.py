"""Host arrays copied to a device in one buffer."""
import numpy as np
import torch

from tnpy_amd.matrix_product_state import upload


def test_upload_views():
    rng = np.random.default_rng(0)
    shapes = [(1, 5, 2, 2), (5, 5, 2, 2), (3,), (7, 1), (0, 4), (5, 1, 2, 2)]
    arrays = [rng.standard_normal(s) for s in shapes]
    arrays.append(np.arange(6).reshape(2, 3).T)  # another type, not contiguous
    out = upload(arrays, torch.device("cpu"))
    for a, t in zip(arrays, out):
        assert t.dtype == torch.float64 and t.is_contiguous() and tuple(t.shape) == a.shape
        assert np.array_equal(t.numpy(), a)
        assert t.storage_offset() % 32 == 0
    assert upload([], torch.device("cpu")) == []
