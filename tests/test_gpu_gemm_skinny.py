"""The Q4_0 products of few activation rows and of row lengths that are no multiple of 256 (csrc/gemm_q4_0_skinny.h):
tile edges, ragged k, every alignment of the weight rows, and the independence of a result from its neighbours.

Bar: both operands are rounded to fp16 (2^-11 each, independent over the products of a sum), the sums are f32: 2e-3 of the largest
result, as for the other prefill kernels.
"""
import numpy as np
import pytest

import oracle
from tests import npref

pytestmark = pytest.mark.gpu
TOL = 2e-3


def _case(seed, m, k, n):
    rng = np.random.default_rng(seed)
    return oracle.quantize_q4_0((rng.standard_normal((n, k)) * 0.02).astype(np.float32)), rng.standard_normal((m, k)).astype(np.float32)


def _run(dev, wq, x, shift=0):
    """The product with the weights `shift` bytes behind a 16-byte boundary."""
    m, k = x.shape
    n = wq.shape[0]
    raw = np.zeros((wq.nbytes + shift + 3) // 4 * 4, np.uint8)
    raw[shift:shift + wq.nbytes] = wq.reshape(-1)
    wb, xb, yb = dev.upload(raw), dev.upload(x), dev.alloc((m * n + 64) * 4)
    dev.upload(np.full(m * n + 64, 7.5, np.float32), yb)
    dev.mul_mat_q4_0_f32(wb.view(shift), xb, yb, k, n, m)
    out = dev.download(yb, np.float32, m * n + 64)
    for b in (wb, xb, yb):
        dev.free(b)
    assert np.all(out[m * n:] == 7.5), "wrote past the end of Y"
    return out[:m * n].reshape(m, n)


@pytest.mark.parametrize("m,k,n", [
    (1, 32, 1), (2, 64, 15), (15, 96, 17), (16, 224, 16), (17, 256, 33), (31, 288, 65), (33, 512, 700), (48, 1024, 4099), (49, 992, 130),
    (64, 3200, 257), (65, 4096, 12288), (80, 2016, 4096), (81, 8224, 96), (97, 8192, 200), (128, 11008, 513), (128, 256, 48),
    (129, 1056, 100), (257, 320, 300), (600, 3200, 131)])
def test_tiles_and_remainders(dev, m, k, n):
    wq, x = _case(m + k + n, m, k, n)
    got = _run(dev, wq, x)
    cols = np.unique(np.concatenate([[0, n - 1], np.random.default_rng(n).choice(n, min(n, 96), replace=False)]))
    emax, el2 = npref.rel_err(got[:, cols], oracle.mul_mat_q4_0_f32(wq[cols], x))
    assert emax < TOL and el2 < TOL, (emax, el2)


@pytest.mark.parametrize("k", [96, 256, 704, 3200])
@pytest.mark.parametrize("m", [5, 70, 150])
def test_the_alignment_of_the_weights_does_not_change_a_bit(dev, m, k):
    """2-byte aligned rows take their blocks apart differently; weights, products and sums stay the same.  (At K = 256
    and 150 rows the 16-byte aligned weights run on the wide kernel, whose sums go in another order.)"""
    wq, x = _case(m * k, m, k, 90)
    ref = _run(dev, wq, x, 4)
    for shift in (2, 6, 8) + (() if k == 256 and m > 80 else (0,)):
        assert np.array_equal(_run(dev, wq, x, shift).view(np.uint32), ref.view(np.uint32)), shift


def test_a_result_does_not_depend_on_its_neighbours(dev):
    """Columns of a wide matrix equal the same rows multiplied as a matrix of their own, rows of a batch the same rows
    in a smaller batch (up to 80 rows, where the wide kernel takes over): tiles, rounds and row blocks change, the order of a
    result's sum does not."""
    wq, x = _case(11, 80, 2048, 6000)
    whole = _run(dev, wq, x)
    assert np.array_equal(whole[:, 333:350], _run(dev, wq[333:350], x))
    assert np.array_equal(whole[:37], _run(dev, wq, x[:37]))


def test_infinities_and_zero_scales_stay_in_their_place(dev):
    """k past the end of a row is padded inside the call: an infinite activation of the last block reaches exactly
    the results that use it, as itself and not as NaN, and none of another row's weights enters."""
    wq, x = _case(5, 20, 288, 40)
    wq = wq.copy()
    wq.reshape(40, 9, 18)[7, :, :2] = 0                       # row 7: scale 0
    wq.reshape(40, 9, 18)[8, :, :2] = np.array([np.inf], np.float16).view(np.uint8)  # row 8: infinite scales
    x[3, 287] = np.inf
    got = _run(dev, wq, x)
    ok = [i for i in range(40) if i not in (7, 8)]
    assert np.all(got[np.arange(20) != 3, 7] == 0) and np.all(np.isfinite(got[np.arange(20) != 3][:, ok]))
    nib = wq.reshape(40, 9, 18)[:, 8, 2 + 15] >> 4            # the weight of k = 287
    for i in ok:
        want = np.nan if nib[i] == 8 else np.inf * np.sign(float(nib[i]) - 8) * np.sign(wq.reshape(40, 9, 18)[i, 8, :2].view(np.float16)[0])
        assert np.isnan(got[3, i]) if np.isnan(want) else got[3, i] == want, i


@pytest.mark.parametrize("m,k,n", [(1, 32, 130), (129, 160, 257), (300, 96, 385), (257, 192, 129), (1100, 288, 4000), (4097, 544, 3001)])
def test_short_rows_and_many_tiles(dev, m, k, n):
    """The sizes that run without a panel (gemm_v1_pays): remainders of its 128 x 128 tiles, weight rows at every 2-byte offset."""
    wq, x = _case(m + k + n, m, k, n)
    got = _run(dev, wq, x)
    cols = np.unique(np.concatenate([[0, n - 1], np.random.default_rng(n).choice(n, min(n, 96), replace=False)]))
    emax, el2 = npref.rel_err(got[:, cols], oracle.mul_mat_q4_0_f32(wq[cols], x))
    assert emax < TOL and el2 < TOL, (emax, el2)
    for shift in (2, 6, 8):
        assert np.array_equal(_run(dev, wq, x, shift).view(np.uint32), got.view(np.uint32)), shift


@pytest.mark.parametrize("m,k,n,shift", [(40, 96, 77, 0), (1, 288, 17, 2), (3, 736, 33, 6), (16, 3200, 131, 0), (17, 8224, 96, 0), (33, 1056, 300, 2),
                                         (150, 992, 257, 0), (130, 512, 200, 2), (65, 11008, 48, 8), (100, 262432, 33, 0), (1600, 11008, 50, 2)])
def test_a_captured_ragged_product_has_the_eager_bits(dev, m, k, n, shift):
    """While a graph is captured nothing is allocated: in a fresh context a product whose K is no multiple of 256, or whose weights
    are not 16-byte aligned, is multiplied in chunks of rows through the context's fixed block (17 MB on 256 compute units: the
    last two cases take several).  Its bits are those of the same call outside a capture, and of a capture that finds the
    workspace large enough."""
    import galois_amd
    d2 = galois_amd.Device(0)
    wq, x = _case(m + k + n, m, k, n)
    want = _run(dev, wq, x, shift)
    emax, el2 = npref.rel_err(want, oracle.mul_mat_q4_0_f32(wq, x))
    assert emax < TOL and el2 < TOL
    raw = np.zeros(wq.nbytes + 16, np.uint8)
    raw[shift:shift + wq.nbytes] = wq.reshape(-1)
    wb, xb, yb = d2.upload(raw), d2.upload(x), d2.alloc((m * n + 64) * 4)
    for warm in (False, True):
        if warm:
            d2.mul_mat_q4_0_f32(wb.view(shift), xb, yb, k, n, m)
        d2.graph_begin_capture()
        d2.mul_mat_q4_0_f32(wb.view(shift), xb, yb, k, n, m)
        g = d2.graph_end_capture()
        for _ in range(3):
            d2.upload(np.full(m * n + 64, 7.5, np.float32), yb)
            d2.graph_launch(g)
            got = d2.download(yb, np.float32, m * n + 64)
            assert np.array_equal(got[:m * n].view(np.uint32), want.reshape(-1).view(np.uint32)), warm
            assert np.all(got[m * n:] == 7.5)
        d2.graph_destroy(g)
    d2.close()


@pytest.mark.parametrize("m,k,n", [(16, 256, 256), (45, 2048, 768), (80, 4096, 2816), (81, 1024, 512), (112, 8192, 256)])
def test_swiglu_and_several_matrices(dev, m, k, n):
    """gate | up with the SwiGLU in the epilogue against the oracle's ops (twice the bar: the result is a product of two), and
    matrices whose boundaries fall inside a tile."""
    (wg, x), (wu, _) = _case(m + n, m, k, n), _case(m + n + 1, m, k, n)
    xb, gb, ub = dev.upload(x), dev.upload(wg), dev.upload(wu)
    pb, po = dev.alloc(dev.f16_panel_bytes(k, m)), dev.alloc(dev.f16_panel_bytes(n, m))
    dev.f32_to_f16_panel(xb, pb, k, m)
    dev.mul_mat_q4_0_swiglu_f16_panel(gb, ub, pb, po, k, n, m)
    t = dev.download(po, np.float16, ((m + 15) // 16, n // 32, 4, 16, 8)).transpose(0, 3, 1, 2, 4).reshape(-1, n)
    want = oracle.mul(oracle.silu(oracle.mul_mat_q4_0_f32(wg, x)).reshape(-1), oracle.mul_mat_q4_0_f32(wu, x).reshape(-1)).reshape(m, n)
    emax, el2 = npref.rel_err(t[:m].astype(np.float32), want)
    assert emax < 2 * TOL and el2 < 2 * TOL and np.all(t[m:] == 0), (emax, el2)
    ns = [3, 18, n - 21]
    ys = [dev.alloc(m * j * 4) for j in ns]
    starts = np.cumsum([0] + ns)
    parts = [dev.upload(np.ascontiguousarray(wg[a:a + j])) for a, j in zip(starts, ns)]
    dev.mul_mat_q4_0_f16_panel(list(zip(parts, ys, ns)), pb, k, m)
    got = np.concatenate([dev.download(y, np.float32, (m, j)) for y, j in zip(ys, ns)], axis=1)
    emax, el2 = npref.rel_err(got, oracle.mul_mat_q4_0_f32(wg, x))
    assert emax < TOL and el2 < TOL, (emax, el2)
    for b in [xb, gb, ub, pb, po] + ys + parts:
        dev.free(b)


@pytest.mark.parametrize("m,n", [(81, 3000), (128, 11008), (129, 5000), (150, 12288), (192, 700), (193, 11008), (300, 12288), (385, 9000), (640, 2000)])
def test_row_tiles_of_the_wide_kernel(dev, m, n):
    """81 rows and up: tiles of 128, 192 or 256 rows and 96 or 48 columns by the workgroups they give.  Against the oracle on a
    sample, and the first 140 rows bit for bit as a batch of their own (another tile, the same order of sums)."""
    k = 512
    wq, x = _case(m + n, m, k, n)
    got = _run(dev, wq, x)
    cols = np.unique(np.concatenate([[0, n - 1], np.random.default_rng(n).choice(n, 96, replace=False)]))
    emax, el2 = npref.rel_err(got[:, cols], oracle.mul_mat_q4_0_f32(wq[cols], x))
    assert emax < TOL and el2 < TOL, (emax, el2)
    if m > 140:
        assert np.array_equal(got[:140].view(np.uint32), _run(dev, wq, x[:140]).view(np.uint32))


@pytest.mark.parametrize("m,k,n", [(100, 8192, 1024), (150, 4096, 768), (190, 1024, 512), (300, 4096, 4096), (390, 2048, 1024),
                                   (447, 8192, 2304), (1400, 4096, 768)])
def test_forms_of_a_narrow_product(dev, m, k, n):
    """With a workspace a narrow product comes whole, in two shares of k or from the few-rows kernel: each sums the same f32
    products in its own order (1e-5 of the largest result)."""
    wq, x = _case(m * 3 + n, m, k, n)
    wb, xb = dev.upload(wq), dev.upload(x)
    pb, ws, y = dev.alloc(dev.f16_panel_bytes(k, m)), dev.alloc(2 * m * n * 4), dev.alloc(m * n * 4)
    dev.f32_to_f16_panel(xb, pb, k, m)
    dev.mul_mat_q4_0_f16_panel([(wb, y, n)], pb, k, m)
    plain = dev.download(y, np.float32, (m, n))
    shares = dev.mul_mat_q4_0_f16_panel_shares(wb, pb, ws, 2 * m * n * 4, k, n, m)
    got = dev.download(ws, np.float32, (2, m, n))[:shares].sum(axis=0)
    assert np.max(np.abs(got - plain)) <= 1e-5 * np.max(np.abs(plain)), shares
    dev.mul_mat_q4_0_f16_panel_add(wb, pb, None, y, k, n, m, ws, 2 * m * n * 4)
    assert np.array_equal(dev.download(y, np.float32, (m, n)), got)
    for b in (wb, xb, pb, ws, y):
        dev.free(b)


@pytest.mark.parametrize("m,k,n", [(81, 8192, 1000), (129, 6400, 48), (200, 8192, 257 * 4), (512, 8192, 2816), (260, 11008, 1536)])
def test_a_large_narrow_product_from_f32_rows(dev, m, k, n):
    """The f32 entry point multiplies these as two shares of k in tiles of 128, 192 or 256 rows: against the oracle on a sample, and
    against the plain panel call, whose sums are one chain (1e-5 of the largest result)."""
    wq, x = _case(m + 2 * n, m, k, n)
    got = _run(dev, wq, x)
    cols = np.unique(np.concatenate([[0, n - 1], np.random.default_rng(n).choice(n, min(n, 96), replace=False)]))
    emax, el2 = npref.rel_err(got[:, cols], oracle.mul_mat_q4_0_f32(wq[cols], x))
    assert emax < TOL and el2 < TOL, (emax, el2)
    wb, xb, pb, y = dev.upload(wq), dev.upload(x), dev.alloc(dev.f16_panel_bytes(k, m)), dev.alloc(m * n * 4)
    dev.f32_to_f16_panel(xb, pb, k, m)
    dev.mul_mat_q4_0_f16_panel([(wb, y, n)], pb, k, m)
    whole = dev.download(y, np.float32, (m, n))
    assert np.max(np.abs(got - whole)) <= 1e-5 * np.max(np.abs(whole))
    assert not np.array_equal(got, whole), "one chain: the call did not come in shares"
    for b in (wb, xb, pb, y):
        dev.free(b)


@pytest.mark.parametrize("m", [81, 128, 129, 192, 193, 260])
def test_swiglu_row_tiles(dev, m):
    k, n = 1024, 2816
    (wg, x), (wu, _) = _case(m, m, k, n), _case(m + 1, m, k, n)
    xb, gb, ub = dev.upload(x), dev.upload(wg), dev.upload(wu)
    pb, po = dev.alloc(dev.f16_panel_bytes(k, m)), dev.alloc(dev.f16_panel_bytes(n, m))
    dev.f32_to_f16_panel(xb, pb, k, m)
    dev.mul_mat_q4_0_swiglu_f16_panel(gb, ub, pb, po, k, n, m)
    t = dev.download(po, np.float16, ((m + 15) // 16, n // 32, 4, 16, 8)).transpose(0, 3, 1, 2, 4).reshape(-1, n)
    want = oracle.mul(oracle.silu(oracle.mul_mat_q4_0_f32(wg, x)).reshape(-1), oracle.mul_mat_q4_0_f32(wu, x).reshape(-1)).reshape(m, n)
    emax, el2 = npref.rel_err(t[:m].astype(np.float32), want)
    assert emax < 2 * TOL and el2 < 2 * TOL and np.all(t[m:] == 0), (emax, el2)
    for b in (xb, gb, ub, pb, po):
        dev.free(b)
