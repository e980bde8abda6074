"""K^T q and V p of one query (the decode step's attention as single ops): the sizes where V p goes from one workgroup's rows to
one launch of sixteen waves to slabs and their sum, columns that end inside a workgroup, and batches in both orders, against f64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f16", [False, True])
@pytest.mark.parametrize("heads, d, rows", [
    (1, 4, 1), (1, 4, 65), (3, 12, 64), (16, 64, 79), (5, 20, 127), (2, 128, 511), (7, 64, 512), (32, 128, 513), (1, 64, 1023), (3, 128, 1024),
    (3, 128, 1025), (9, 32, 2000)])
def test_products_of_one_query(dev, heads, d, rows, f16):
    print(heads, d, rows, f16, flush=True)
    rng = np.random.default_rng(heads * rows + d)
    e = heads * d
    ct = np.float16 if f16 else np.float32
    mul = dev.mul_mat_f16_f32 if f16 else dev.mul_mat_f32
    cache = rng.standard_normal((rows, e)).astype(ct)              # [position][head * d], as the caches lie
    p = rng.random((heads, rows)).astype(np.float32)
    q = rng.standard_normal((heads, d)).astype(np.float32)
    cb, pb, qb = dev.upload(cache), dev.upload(p), dev.upload(q)
    out, s = dev.upload(np.full(e + 64, 7.5, np.float32)), dev.upload(np.full(heads * rows + 64, 7.5, np.float32))
    c64 = cache.astype(np.float64).reshape(rows, heads, d)
    # V p: V seen as [rows, d, heads] with strides (e, 1, d)
    mul(cb, pb, out, rows, d, 1, heads, heads, e, 1, d)
    got = dev.download(out, np.float32, e + 64)
    want = np.einsum("lhd,hl->hd", c64, p.astype(np.float64))
    bound = 2.0 ** -23 * (np.sqrt(rows) + 4) * 4 * np.sqrt(np.einsum("lhd,hl->hd", c64 ** 2, p.astype(np.float64) ** 2)) + 1e-30
    assert np.all(np.abs(got[:e].reshape(heads, d) - want) <= bound) and np.all(got[e:] == 7.5)
    # K^T q: K seen as [d, rows, heads] with strides (1, e, d)
    mul(cb, qb, s, d, rows, 1, heads, heads, 1, e, d)
    got = dev.download(s, np.float32, heads * rows + 64)
    want = np.einsum("lhd,hd->hl", c64, q.astype(np.float64))
    bound = 2.0 ** -23 * (np.sqrt(d) + 4) * 4 * np.sqrt(np.einsum("lhd,hd->hl", c64 ** 2, q.astype(np.float64) ** 2)) + 1e-30
    assert np.all(np.abs(got[:heads * rows].reshape(heads, rows) - want) <= bound) and np.all(got[heads * rows:] == 7.5)
    for b in (cb, pb, qb, out, s):
        dev.free(b)
