"""Two int32 values to the device in stream order (galois_hip_store_i32_pair): the words, their neighbours, and the refusals."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_two_values_in_stream_order(dev):
    b = dev.upload(np.arange(4, dtype=np.int32))
    dev._check(dev._lib.galois_hip_store_i32_pair(dev._ctx, b.ptr, -7, b.ptr + 12, 1 << 30))
    assert dev.download(b, np.int32, 4).tolist() == [-7, 1, 2, 1 << 30]
    assert dev._lib.galois_hip_store_i32_pair(dev._ctx, None, 1, b.ptr, 1) == -1
    assert dev._lib.galois_hip_store_i32_pair(dev._ctx, b.ptr + 2, 1, b.ptr, 1) == -3
    dev.free(b)
