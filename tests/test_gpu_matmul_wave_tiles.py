"""The f32 matrix-core products at the edges of their tiles: 32 rows of b, 64 columns, chunks of 16 k dealt to four waves --
against the oracle through the cases of test_gpu_matmul_prefill_attn (scores and V p of the same sizes)."""
import pytest

from tests import test_gpu_matmul_prefill_attn as cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,H,D,M", [(1, 2, 64, 16), (15, 1, 64, 31), (16, 3, 64, 32), (17, 2, 80, 33), (63, 2, 63, 64), (64, 1, 65, 65),
                                     (65, 2, 128, 16), (80, 1, 130, 40), (127, 3, 8, 20), (129, 1, 64, 129), (257, 2, 33, 47)])
@pytest.mark.parametrize("f16", [False, True])
def test_tile_edges(dev, L, H, D, M, f16):
    cases.test_prefill_attention_products(dev, L, H, D, M, f16)
