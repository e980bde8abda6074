"""The decode attention at the lines between its workgroup shapes (64, 128 or 256 keys, 256 or 512 threads; csrc/attn_decode.hip)
and of its merge (one split, up to 16, 24, 32, more), against the op sequence of test_gpu_attn."""
import pytest

from tests import test_gpu_attn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,D,keys", [
    (32, 128, 64), (32, 128, 192), (32, 128, 193), (32, 128, 256), (32, 128, 257), (32, 128, 512), (32, 128, 513), (32, 128, 2049),
    (8, 128, 1024), (8, 128, 1025), (5, 128, 4096), (5, 128, 4097), (64, 128, 1100), (2, 64, 128), (2, 64, 129), (2, 64, 256),
    (2, 64, 257), (3, 64, 2048), (3, 64, 2049), (3, 64, 4200), (3, 64, 8300), (2, 128, 3072), (2, 128, 3073),
    (2, 64, 6144), (2, 64, 6145), (64, 64, 2100), (64, 64, 2600)])
@pytest.mark.parametrize("f16", [False, True])
def test_workgroup_shapes(dev, H, D, keys, f16):
    check = test_gpu_attn.test_attn_decode_with_f16_caches if f16 else test_gpu_attn.test_attn_decode_matches_the_op_sequence
    check(dev, H, D, keys + 3, keys - 1)
