"""The prefill attention with its keys split over several workgroups (few rows behind a long context) against the op sequence in
f64 of test_gpu_attn_prefill: row counts around a tile, contexts that divide into stages unevenly, walks shorter than the
number of splits, both caches, both outputs; and the same bits in a fresh context, in a used one and in a capture."""
import numpy as np
import pytest

from tests import npref
from tests import test_gpu_attn_prefill as whole

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv_f16", [False, True])
@pytest.mark.parametrize("n_head,n,n_past", [(2, 1, 700), (1, 9, 1900), (3, 16, 1023), (2, 17, 1024), (2, 63, 1601), (2, 64, 960),
                                             (1, 65, 959), (5, 150, 1201), (2, 700, 300), (1, 1000, 0), (32, 9, 640), (2, 200, 4000)])
def test_split_keys_against_the_op_sequence_in_f64(dev, n_head, n, n_past, kv_f16):
    whole.test_attention_of_many_rows_against_the_op_sequence_in_f64(dev, n_head, n, n_past, kv_f16)


@pytest.mark.parametrize("n_head,n,n_past,kv_f16", [(2, 20, 1500, False), (32, 150, 1201, True), (1, 1000, 0, False)])
def test_the_bits_do_not_depend_on_what_ran_before(dev, n_head, n, n_past, kv_f16):
    """A call captured as the first one of a fresh context, captured again after another call has grown the context's workspace, and
    issued outside a capture: the same bits (whether the keys are split is decided by sizes alone)."""
    import galois_amd
    d2 = galois_amd.Device(0)
    q, kc, vc = whole._inputs(7, n_head, n, n_past, n_past + n, kv_f16)
    scale = float(np.float32(128) ** np.float32(-0.5))
    ref = whole._reference(q, kc, vc, n_head, n_past, scale)
    nb = n * n_head * 128
    qb, kb, vb, ob = d2.upload(q), d2.upload(kc), d2.upload(vc), d2.alloc(nb * 4)
    wb, xb, yb = d2.alloc(2048 * 144), d2.alloc(2048 * 256 * 4), d2.alloc(2048 * 2048 * 4)
    got = []
    for warm in (False, True):
        if warm:    # a product of 2048 rows: the workspace grows
            d2.mul_mat_q4_0_f32(wb, xb, yb, 256, 2048, 2048)
        d2.graph_begin_capture()
        d2.attn_prefill(qb, kb, vb, ob, None, n_head, 128, n, n_past, scale, kv_f16=kv_f16)
        g = d2.graph_end_capture()
        for _ in range(3):
            d2.upload(np.zeros(nb, np.float32), ob)
            d2.graph_launch(g)
            got.append(d2.download(ob, np.float32, (n, n_head * 128)))
        d2.graph_destroy(g)
    d2.attn_prefill(qb, kb, vb, ob, None, n_head, 128, n, n_past, scale, kv_f16=kv_f16)
    got.append(d2.download(ob, np.float32, (n, n_head * 128)))
    emax, el2 = npref.rel_err(got[0], ref)
    assert emax < whole.TOL and el2 < whole.TOL
    for o in got[1:]:
        assert np.array_equal(o.view(np.uint32), got[0].view(np.uint32))
    d2.close()
