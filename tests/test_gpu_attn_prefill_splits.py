"""The prefill attention with its keys split over several workgroups (few rows behind a long context) against the op sequence in
f64 of test_gpu_attn_prefill: row counts around a tile, contexts that divide into stages unevenly, walks shorter than the
number of splits, both caches, both outputs; and during a graph capture, where a context without a workspace keeps the keys
whole."""
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


def test_a_capture_without_a_workspace_keeps_the_keys_whole(dev):
    import galois_amd
    d2 = galois_amd.Device(0)
    n_head, n, n_past = 2, 20, 1500
    q, kc, vc = whole._inputs(7, n_head, n, n_past, n_past + n, False)
    scale = float(np.float32(128) ** np.float32(-0.5))
    ref = whole._reference(q, kc, vc, n_head, n_past, scale)
    qb, kb, vb, ob = d2.upload(q), d2.upload(kc), d2.upload(vc), d2.alloc(n * n_head * 128 * 4)
    for warm in (False, True):
        if warm:    # outside a capture the workspace grows, and the next capture splits the keys
            d2.attn_prefill(qb, kb, vb, ob, None, n_head, 128, n, n_past, scale)
        d2.graph_begin_capture()
        d2.attn_prefill(qb, kb, vb, ob, None, n_head, 128, n, n_past, scale)
        g = d2.graph_end_capture()
        for _ in range(3):
            d2.upload(np.zeros(n * n_head * 128, np.float32), ob)
            d2.graph_launch(g)
            emax, el2 = npref.rel_err(d2.download(ob, np.float32, (n, n_head * 128)), ref)
            assert emax < whole.TOL and el2 < whole.TOL
        d2.graph_destroy(g)
    for b in (qb, kb, vb, ob):
        d2.free(b)
    d2.close()
