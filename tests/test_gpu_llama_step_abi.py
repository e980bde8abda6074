"""galois_hip_llama_step through the C ABI itself: what it refuses (before anything is launched: token, position and logits stay
as they are), and a token and position that lie on the device, one outside the vocabulary among them."""
import ctypes as C

import numpy as np
import pytest

from galois_amd import _abi

pytestmark = pytest.mark.gpu

E, H, F, V, LAYERS, CTX = 512, 4, 576, 300, 2, 140
E_NULL, E_SHAPE, E_ALIGN, E_UNSUPPORTED = -1, -2, -3, -5


def _q4(rng, n, k):
    b = rng.integers(0, 256, (n, k // 32, 18), dtype=np.uint8)
    b[..., :2] = (0.004 + 0.002 * rng.random((n, k // 32))).astype(np.float16)[..., None].view(np.uint8)
    return b.reshape(-1)


class _Model:
    """A model's buffers behind the struct the call takes."""

    def __init__(self, dev, seed=0, kv_f16=False):
        rng = np.random.default_rng(seed)
        self.dev, self.bufs = dev, []
        self.layers = (_abi.LlamaLayer * LAYERS)()
        for y in self.layers:
            for name, (n, k) in dict(wq=(E, E), wk=(E, E), wv=(E, E), wo=(E, E), w_gate=(F, E), w_up=(F, E), w_down=(E, F)).items():
                setattr(y, name, self._up(_q4(rng, n, k)))
            y.attn_norm, y.ffn_norm = (self._up((1 + 0.1 * rng.standard_normal(E)).astype(np.float32)) for _ in range(2))
            y.k_cache, y.v_cache = (self._up(rng.standard_normal((CTX, E)).astype(np.float16 if kv_f16 else np.float32)) for _ in range(2))
        m = self.m = _abi.LlamaModel(n_embd=E, n_head=H, n_ff=F, n_vocab=V, n_layer=LAYERS, n_ctx=CTX, kv_f16=int(kv_f16), rms_eps=1e-6,
                                     freq_scale=1.0, theta_scale=10000.0 ** (-2.0 / 128), scale=128 ** -0.5, layers=self.layers)
        m.tok_embd, m.output = self._up(_q4(rng, V, E)), self._up(_q4(rng, V, E))
        m.out_norm = self._up((1 + 0.1 * rng.standard_normal(E)).astype(np.float32))
        m.logits, m.token, m.pos = self._up(np.full(V, 7.5, np.float32)), self._up(np.int32([-9])), self._up(np.int32([-9]))
        bytes_ = C.c_int64()
        dev._check(dev._lib.galois_hip_llama_step_workspace(dev._ctx, C.byref(m), C.byref(bytes_)))
        assert bytes_.value > 0
        m.workspace, m.workspace_bytes = self._up(np.zeros(bytes_.value, np.uint8)), bytes_.value

    def _up(self, a):
        self.bufs.append(self.dev.upload(a))
        return self.bufs[-1].ptr

    def step(self, token, n_past):
        return self.dev._lib.galois_hip_llama_step(self.dev._ctx, C.byref(self.m), token, n_past)

    def get(self, field, dtype, shape):
        ptr = getattr(self.m, field)
        return self.dev.download(next(b for b in self.bufs if b.ptr == ptr), dtype, shape)

    def close(self):
        for b in self.bufs:
            self.dev.free(b)


def test_what_the_call_refuses(dev):
    mo = _Model(dev)
    m, n_past = mo.m, 20
    ok = {f: getattr(m, f) for f, _ in m._fields_}

    def refused(status, fields={}, token=5, past=n_past):
        for f, v in fields.items():
            setattr(m, f, v)
        assert mo.step(token, past) == status, (fields, token, past)
        for f in fields:
            setattr(m, f, ok[f])

    # capacities of a head that do not hold row n_past: the row would land in the next head, the last head's past the cache
    for n in (-1, -CTX, 1, n_past, -(1 << 31)):
        refused(E_SHAPE, dict(head_major_n_ctx=n))
    refused(E_SHAPE, past=CTX)
    refused(E_SHAPE, past=-1)
    refused(E_SHAPE, token=V)
    refused(E_SHAPE, dict(workspace_bytes=ok["workspace_bytes"] - 1))
    for f in ("tok_embd", "output", "out_norm", "logits", "token", "pos", "workspace"):
        refused(E_NULL, {f: None})
    for f, off in (("tok_embd", 1), ("output", 2), ("out_norm", 4), ("logits", 2), ("token", 2), ("pos", 2), ("workspace", 128)):
        refused(E_ALIGN, {f: ok[f] + off})
    for fields in (dict(n_head=8), dict(n_embd=4224, n_head=33), dict(n_ff=F + 32), dict(n_ff=12352), dict(n_layer=251), dict(n_vocab=(1 << 24) + 1)):
        refused(E_UNSUPPORTED, fields)
    y = mo.layers[1]
    for f, off, status in (("wq", None, E_NULL), ("w_down", 2, E_ALIGN), ("ffn_norm", 4, E_ALIGN), ("v_cache", 8, E_ALIGN), ("k_cache", None, E_NULL)):
        keep = getattr(y, f)
        setattr(y, f, None if off is None else keep + off)
        assert mo.step(5, n_past) == status, f
        setattr(y, f, keep)
    dev.synchronize()
    assert mo.get("token", np.int32, 1)[0] == -9 and mo.get("pos", np.int32, 1)[0] == -9
    assert np.all(mo.get("logits", np.float32, V) == 7.5)
    # and it takes the same model again, also with the smallest capacity of a head that holds the row
    assert mo.step(5, n_past) == 0
    assert np.all(np.isfinite(mo.get("logits", np.float32, V)))
    m.head_major_n_ctx = n_past + 1
    assert mo.step(5, n_past) == 0
    assert np.all(np.isfinite(mo.get("logits", np.float32, V)))
    mo.close()


def test_token_and_position_on_the_device(dev):
    """token < 0: those the device holds, the same bits as passed by value; a token outside the vocabulary gives NaN and no more."""
    mo = _Model(dev, seed=1, kv_f16=True)
    assert mo.step(17, 130) == 0
    want = mo.get("logits", np.float32, V)
    assert mo.get("token", np.int32, 1)[0] == 17 and mo.get("pos", np.int32, 1)[0] == 130 and np.all(np.isfinite(want))
    token = next(b for b in mo.bufs if b.ptr == mo.m.token)
    for t in (V, -1, 0x7FFFFFFF):
        dev.upload(np.int32([t]), token)
        assert mo.step(-1, 130) == 0
        assert np.all(np.isnan(mo.get("logits", np.float32, V)))
    dev.upload(np.int32([17]), token)
    for _ in range(3):
        assert mo.step(-1, 130) == 0
        assert np.array_equal(mo.get("logits", np.float32, V), want)
    mo.close()
