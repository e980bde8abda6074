"""The decode step in one grid against the oracle's op-by-op step: from an empty cache over several tokens, on filled caches in
every layout and type, where a split of the keys ends, and from a graph.  (Models narrower than 512 columns do not take the grid.)"""
import numpy as np
import pytest

from galois_amd import host_api as g
from tests.test_gpu_llama import _check, _load, _make_weights, _ref_step

pytestmark = pytest.mark.gpu

HP = dict(n_vocab=515, n_embd=512, n_head=4, n_layer=3, n_ff=832, n_ctx=300, rms_eps=1e-6, freq_base=10000.0)
TOL = {False: 1e-4, True: 2e-4}   # one matvec's bar; rows that an f16 cache rounds may fall to the other side


@pytest.fixture(scope="module")
def gdev():
    return g.Device.gpu(0)


@pytest.mark.parametrize("kv_f16, head_major", [(False, False), (False, True), (True, False), (True, True)])
def test_from_an_empty_cache_over_several_tokens(gdev, kv_f16, head_major):
    w = _make_weights(np.random.default_rng(71), HP)
    dec = g.LlamaDecoder(gdev, kv_f16=kv_f16, kv_head_major=head_major, **HP)
    _load(dec, w)
    kc = np.zeros((HP["n_layer"], HP["n_ctx"], HP["n_embd"]), np.float32)
    vc = np.zeros_like(kc)
    toks = [1, 400, 17, 17, 514, 0, 250, 3, 77]
    for n_past, tok in enumerate(toks):
        ref = _ref_step(w, HP, kc, vc, tok, n_past, round_kv=kv_f16)
        dec.decode(tok, n_past, 5)
        assert dec.calls_per_step() == 1
        _check(dec.logits(), ref, TOL[kv_f16])
    n = len(toks)
    for i in range(HP["n_layer"]):
        for name, want in (("k_cache", kc), ("v_cache", vc)):
            got = dec.tensor(name, i).to_cpu_tensor().astype(np.float32)
            if head_major:
                got = got.transpose(1, 0, 2).reshape(HP["n_ctx"], -1)
            assert not got[n:].any()
            _check(got[:n], want[i][:n], 1e-3 if kv_f16 else 1e-4)
    dec.close()


@pytest.mark.parametrize("n_past", [127, 128, 255, 256, 299])
@pytest.mark.parametrize("kv_f16, head_major", [(False, False), (False, True), (True, False), (True, True)])
def test_on_filled_caches_and_from_a_graph(gdev, kv_f16, head_major, n_past):
    rng = np.random.default_rng(72)
    w = _make_weights(rng, HP)
    ct = np.float16 if kv_f16 else np.float32
    shape = (HP["n_layer"], HP["n_ctx"], HP["n_embd"])
    kc, vc = rng.standard_normal(shape).astype(ct), rng.standard_normal(shape).astype(ct)
    dec = g.LlamaDecoder(gdev, kv_f16=kv_f16, kv_head_major=head_major, **HP)
    ref = _ref_step(w, HP, kc.astype(np.float32), vc.astype(np.float32), 123, n_past, round_kv=kv_f16)
    _load(dec, w, kc, vc)
    dec.decode(123, n_past, 5)
    assert dec.calls_per_step() == 1
    eager = dec.logits().copy()
    _check(eager, ref, TOL[kv_f16])
    dec.capture(123, n_past, 5)
    for _ in range(3):
        _load(dec, w, kc, vc)
        dec.replay()
        assert np.array_equal(dec.logits(), eager)
        dec.decode(5, n_past - 1, 5)
        dec.decode(123, n_past, 5)
    dec.close()
