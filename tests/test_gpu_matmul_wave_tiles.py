"""The f32 matrix-core products at the edges of their tiles: 32 rows of b, 64 columns, chunks of 16 k dealt to four waves --
against the oracle through the cases of test_gpu_matmul_prefill_attn (scores and V p of the same sizes)."""
import numpy as np
import pytest

from tests import test_gpu_matmul_prefill_attn as cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L,H,D,M", [(1, 2, 64, 16), (15, 1, 64, 31), (16, 3, 64, 32), (17, 2, 80, 33), (63, 2, 63, 64), (64, 1, 65, 65),
                                     (65, 2, 128, 16), (80, 1, 130, 40), (127, 3, 8, 20), (129, 1, 64, 129), (257, 2, 33, 47)])
@pytest.mark.parametrize("f16", [False, True])
def test_tile_edges(dev, L, H, D, M, f16):
    cases.test_prefill_attention_products(dev, L, H, D, M, f16)


@pytest.mark.parametrize("K,N,M,B", [(16, 64, 16, 1), (17, 33, 31, 3), (40, 300, 500, 8), (33, 1000, 130, 16), (100, 4099, 257, 2), (64, 64, 2048, 32),
                                     (128, 2048, 512, 8), (500, 130, 40, 2)])
@pytest.mark.parametrize("f16", [False, True])
def test_a_contiguous_along_n_split_and_whole(dev, K, N, M, B, f16):
    """Either side of the rule that deals K to a workgroup's waves.  Every result of K f32 products is within (K + 2) 2^-24 of the sum
    of their magnitudes, whatever the order they are added in."""
    rng = np.random.default_rng(K + N)
    a = rng.standard_normal((B, K, N)).astype(np.float16 if f16 else np.float32)
    b = rng.standard_normal((B, M, K)).astype(np.float32)
    ab, bb, db = dev.upload(a), dev.upload(b), dev.upload(np.full(B * M * N + 64, 7.5, np.float32))
    (dev.mul_mat_f16_f32 if f16 else dev.mul_mat_f32)(ab, bb, db, K, N, M, B, B, N, 1, K * N)
    got = dev.download(db, np.float32, B * M * N + 64)
    assert np.all(got[B * M * N:] == 7.5)
    a, b = a.astype(np.float64), b.astype(np.float64)
    for i in {0, B - 1}:
        err = np.abs(got[i * M * N:(i + 1) * M * N].reshape(M, N) - b[i] @ a[i])
        assert np.all(err <= (K + 2) * 2.0 ** -24 * (np.abs(b[i]) @ np.abs(a[i])))
    for buf in (ab, bb, db):
        dev.free(buf)


def test_more_workgroups_than_a_launch_holds_along_x(dev):
    """16 rows of more than 2^30 columns: over 2^32 threads, so the workgroups go on along z.  K = 1: every result is one product."""
    N, M = (1 << 30) + 4099, 16
    row = np.random.default_rng(0).standard_normal(1 << 20).astype(np.float32)
    a, d = dev.alloc(N * 4), dev.alloc((N * M + 64) * 4)
    dev.upload(row, a)
    have = row.size
    while have < N:
        n = min(have, N - have)
        dev.copy_d2d(a.view(have * 4), a, n * 4)
        have += n
    b = np.arange(1, M + 1, dtype=np.float32)
    bb = dev.upload(b)
    dev.mul_mat_f32(a, bb, d, 1, N, M, 1, 1, N, 1, N)
    for m in (0, 7, 15):
        for at in (0, (1 << 29) - 1000, N - 70000):
            n = 70000
            got = dev.download(d.view((m * N + at) * 4), np.float32, n)
            assert np.array_equal(got, b[m] * row[(at + np.arange(n)) % row.size])
    assert np.all(dev.download(d.view(N * M * 4), np.float32, 64) == 0)
    for buf in (a, d, bb):
        dev.free(buf)
