"""q | k | v of a prefill with the rotations and the append in the products' epilogue (galois_hip_mul_mat_q4_0_qkv_rope_f16_panel)
against the two calls it replaces: the same bits, on the few-rows kernel (up to 80 rows) and on every tile of the wide one, for
f32 and f16 cache rows, at the edges of row tiles and of the column tiles that reach over a matrix's end."""
import numpy as np
import pytest

from galois_amd import GaloisHipError

pytestmark = pytest.mark.gpu
THETA = float(np.float32(10000.0) ** np.float32(-2.0 / 128))


def _q4(rng, n, k):
    b = rng.integers(0, 256, (n, k // 32, 18), dtype=np.uint8)
    b[..., :2] = (0.01 * rng.standard_normal((n, k // 32))).astype(np.float16)[..., None].view(np.uint8)
    return b.reshape(-1)


# heads: 1 and 3 end tiles of 48, 64 (rows per wave) and 96 columns inside a matrix; 32 x 512 rows are whole tiles of 96 x 256
@pytest.mark.parametrize("heads, k, m, first", [
    (1, 256, 1, 0), (1, 512, 16, 5), (3, 256, 17, 4000), (3, 2304, 80, 1), (2, 8192, 40, 9), (20, 2560, 23, 77), (86, 256, 70, 3),
    (1, 256, 81, 2), (3, 512, 129, 0), (5, 256, 192, 1201), (20, 512, 150, 30), (32, 4096, 300, 0), (32, 4096, 512, 1536), (9, 1024, 1000, 1)])
@pytest.mark.parametrize("kv_f16", [False, True])
def test_same_bits_as_the_two_calls(dev, heads, k, m, first, kv_f16):
    print(heads, k, m, first, kv_f16, flush=True)
    rng = np.random.default_rng(heads * k + m)
    e = heads * 128
    w = [dev.upload(_q4(rng, e, k)) for _ in range(3)]
    x = dev.upload(rng.standard_normal((m, k)).astype(np.float32))
    panel = dev.alloc(dev.f16_panel_bytes(k, m))
    dev.f32_to_f16_panel(x, panel, k, m)
    ct, size = (np.float16, 2) if kv_f16 else (np.float32, 4)
    q, kk, v, qr = (dev.alloc(m * e * 4) for _ in range(4))
    guard = 64
    want_k, want_v, got_k, got_v, got_q = (dev.upload(np.full(m * e + guard, 7.5, t)) for t in (ct, ct, ct, ct, np.float32))
    pos = dev.upload(np.arange(first, first + m, dtype=np.int32))
    pairs = dev.alloc(m * 128 * 4)
    dev.mul_mat_q4_0_f16_panel([(w[0], q, e), (w[1], kk, e), (w[2], v, e)], panel, k, m)
    dev.rope_qk_append(q, kk, v, qr, want_k, want_v, kv_f16, 128, heads, m, pos, 1.0, THETA)
    dev.rope_pairs(pairs, m, first, 1.0, THETA)
    dev.mul_mat_q4_0_qkv_rope_f16_panel(w[0], w[1], w[2], panel, pairs, got_q, got_k, got_v, kv_f16, 128, heads, k, m)
    bits = np.uint16 if kv_f16 else np.uint32
    assert np.array_equal(dev.download(got_q, np.uint32, m * e + guard)[:m * e], dev.download(qr, np.uint32, m * e))
    for got, want in ((got_k, want_k), (got_v, want_v)):
        assert np.array_equal(dev.download(got, bits, m * e + guard), dev.download(want, bits, m * e + guard))
    assert np.all(dev.download(got_q, np.float32, m * e + guard)[m * e:] == 7.5), "wrote past the end of q"
    for b in [x, panel, q, kk, v, qr, want_k, want_v, got_k, got_v, got_q, pos, pairs] + w:
        dev.free(b)


def test_refusals(dev):
    b = dev.alloc(1 << 16)
    for args, status in (((False, 64, 2, 256, 1), -5), ((False, 128, 0, 256, 1), -2), ((False, 128, 1, 128, 1), -2), ((False, 128, 1, 256, 0), -2)):
        with pytest.raises(GaloisHipError) as ei:
            dev.mul_mat_q4_0_qkv_rope_f16_panel(b, b, b, b, b, b, b, b, *args)
        assert ei.value.status == status
    for args in ((0, 0), (1, -1), ((1 << 24) + 1, 0), (2, 0x7FFFFFFE)):
        with pytest.raises(GaloisHipError) as ei:
            dev.rope_pairs(b, *args, 1.0, THETA)
        assert ei.value.status == -2
    dev.free(b)
