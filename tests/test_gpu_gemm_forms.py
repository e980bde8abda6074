"""The few-rows matmul's weights as whole runs of their rows, as slots and as blocks, and its tiles of one to four weight
tiles: a result does not depend on the columns around it, so a wide product (which takes runs, and three or four tiles a
wave) has the bits of the same columns multiplied a few at a time (slots, one tile), at the edges of pieces, tiles and rows;
and both agree with the product in f64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _weights(rng, n, k):
    b = rng.integers(0, 256, (n, k // 32, 18), dtype=np.uint8)
    b[..., :2] = (0.01 * rng.standard_normal((n, k // 32))).astype(np.float16)[..., None].view(np.uint8)
    return b


def _dequant(b):
    d = b[..., :2].copy().view(np.float16)[..., 0].astype(np.float64)
    q = np.concatenate([b[..., 2:] & 15, b[..., 2:] >> 4], axis=-1).astype(np.float64) - 8
    # each weight is rounded to fp16 once, as the matrix cores take it
    return (q * d[..., None]).astype(np.float16).astype(np.float64).reshape(b.shape[0], -1)


# 8200 columns: 171 workgroups of three tiles, 513 of one; 12288: 256 of three; 3000: 188 of one; 40000: several rounds of four
@pytest.mark.parametrize("k, n, ms", [
    (2304, 8200, (1, 16, 17, 33, 64, 80)),     # nine pieces of 256: waves with two and three
    (256, 12288, (5, 48)),                      # one piece: three of the four waves have none
    (8192, 3000, (3, 40, 77)),                  # eight waves a workgroup, runs at any width
    (8192, 6752, (52, 64)),                     # tiles of two by four
    (8448, 8209, (20,)),
    (3200, 8640, (2, 77)),                      # rows that are not whole pieces: slots
    (2400, 8640, (18, 50)),                     # an odd number of blocks
    (1024, 40000, (9, 30)),
])
def test_wide_products_have_the_bits_of_their_columns(dev, k, n, ms):
    rng = np.random.default_rng(k + n)
    w = _weights(rng, n, k)
    wb = dev.upload(w.reshape(-1))
    row = k // 32 * 18
    step = 48
    some = [0, (n // 2 + 15) // 16 * 16, n - step]      # columns looked at one narrow product at a time
    ref_w = {c: _dequant(w[c:c + step]) for c in some}
    for m in ms:
        print(k, n, m, flush=True)
        x = rng.standard_normal((m, k)).astype(np.float32)
        xb, yb, zb = dev.upload(x), dev.alloc(m * n * 4), dev.alloc(m * step * 4)
        dev.mul_mat_q4_0_f32(wb, xb, yb, k, n, m)
        y = dev.download(yb, np.float32, (m, n))
        for c in some:
            dev.mul_mat_q4_0_f32(wb.view(c * row), xb, zb, k, step, m)
            assert np.array_equal(dev.download(zb, np.float32, (m, step)), y[:, c:c + step]), (m, c)
            ref = x.astype(np.float16).astype(np.float64) @ ref_w[c].T
            # operands are the reference's; k f32 additions of products of size |x| |w|
            bound = 2.0 ** -23 * k ** 0.5 * 8 * np.linalg.norm(x, axis=1)[:, None] * np.linalg.norm(ref_w[c], axis=1)[None]
            assert np.all(np.abs(y[:, c:c + step] - ref) <= bound), (m, c)
        for b in (xb, yb, zb):
            dev.free(b)
    dev.free(wb)


@pytest.mark.parametrize("k, n", [(1024, 12288), (2304, 12800), (8192, 16384)])
def test_four_weight_tiles_by_four_row_tiles(dev, k, n):
    """49 to 64 rows of 12288 to 16384 columns: the widest tiles a wave has, with four and with eight waves a workgroup."""
    test_wide_products_have_the_bits_of_their_columns(dev, k, n, (49, 63, 64))
