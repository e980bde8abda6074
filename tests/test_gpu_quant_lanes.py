"""The two quantizer kernels (eight lanes a block for 16-byte aligned arrays, a thread a block otherwise) give the oracle's
bytes, at the edges of a workgroup's 128 blocks and for the values where a rule could be told apart: ties of magnitude
between lanes, zeros of either sign, tiny and huge blocks."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _blocks(nb, seed):
    rng = np.random.default_rng(seed)
    x = (rng.standard_normal((nb, 32)) * np.exp(rng.uniform(-8, 8, (nb, 1)))).astype(np.float32)
    for b in range(0, nb, 3):  # ties: the largest magnitude again elsewhere with the other sign
        i, j = rng.choice(32, 2, replace=False)
        x[b, i] = np.abs(x[b]).max() * 1.5
        x[b, j] = -x[b, i]
    if nb > 8:
        x[1], x[2], x[4] = 0.0, -0.0, 1e-36 * rng.standard_normal(32)
        x[5, 7] = 3e38
    return x


@pytest.mark.parametrize("nb", [1, 2, 31, 32, 33, 127, 128, 129, 255, 257, 1000, 4099])
@pytest.mark.parametrize("shift", [0, 1])
def test_bytes_and_values(dev, nb, shift):
    x = _blocks(nb, nb)
    want = oracle.quantize_q4_0(x).reshape(-1)
    xb, qb = dev.alloc(x.nbytes + 16), dev.upload(np.full((want.nbytes + 67) // 4 * 4, 0xA5, np.uint8))
    yb = dev.upload(np.full(nb * 32 + 20, 7.5, np.float32))
    dev.upload(np.concatenate([np.zeros(shift, np.float32), x.reshape(-1)]), xb)
    q = qb.view(2 * shift)
    dev.quantize_row_q4_0(xb.view(4 * shift), q, x.size)
    got = dev.download(qb, np.uint8, qb.nbytes)[2 * shift:]
    assert np.array_equal(got[:want.nbytes], want)
    assert np.all(got[want.nbytes:] == 0xA5)
    dev.dequantize_row_q4_0(q, yb.view(4 * shift), x.size)
    y = dev.download(yb, np.float32, nb * 32 + 20)[shift:]
    assert np.array_equal(y[:x.size].view(np.uint32), oracle.dequantize_q4_0(want.reshape(nb, 18)).reshape(-1).view(np.uint32))
    assert np.all(y[x.size:] == 7.5)
    for b in (xb, qb, yb):
        dev.free(b)


def test_non_finite_blocks_agree_between_the_kernels(dev):
    """What the rule leaves to the conversion instructions (NaN and infinity to an integer: non-finite values, and blocks so
    small that the reciprocal of their scale overflows, below 2^-125) is the same in both."""
    x = _blocks(300, 9)
    x[4], x[8] = 1e-41 * np.arange(32), -1e-39
    x[::2, 3], x[1::4, 17], x[3::4, 30] = np.inf, np.nan, -np.inf
    xb, xs = dev.upload(x), dev.alloc(x.nbytes + 16)
    dev.upload(np.concatenate([np.zeros(1, np.float32), x.reshape(-1)]), xs)
    qa, qs = dev.alloc(300 * 18 + 8), dev.alloc(300 * 18 + 8)
    dev.quantize_row_q4_0(xb, qa, x.size)
    dev.quantize_row_q4_0(xs.view(4), qs, x.size)
    assert np.array_equal(dev.download(qa, np.uint8, 5400), dev.download(qs, np.uint8, 5400))
    for b in (xb, xs, qa, qs):
        dev.free(b)
