"""The decode step that goes out as one call (galois_hip_llama_step, launch plan 5 where it takes the model) against the
plan that issues it launch by launch (plan 4), at the sizes where its dispatch changes: one workgroup's rows left over in a
stage, vectors of one, two and three chunks, the edges of a key split, the first and last number of splits, more layers
than a launch carries; recorded, repeated and interleaved; and with its in-launch waits running out."""
import numpy as np
import pytest

from galois_amd import host_api as g

pytestmark = pytest.mark.gpu

BASE = dict(n_vocab=515, n_embd=512, n_head=4, n_layer=2, n_ff=512, n_ctx=160, rms_eps=1e-6, freq_base=10000.0)
# both plans round activations to 18 bits of their block and add f32 in other orders: 1e-5 a product, a few of them a layer;
# an f16 cache row may differ by a unit in the last place where that falls on the other side (2^-11 of one element)
TOL = {False: 1e-4, True: 4e-4}


@pytest.fixture(scope="module")
def gdev():
    return g.Device.gpu(0)


def _q4(rng, n, k):
    """Random Q4_0 blocks: f16 scales about 0.005, nibbles uniform."""
    b = rng.integers(0, 256, (n, k // 32, 18), dtype=np.uint8)
    b[..., :2] = (0.004 + 0.002 * rng.random((n, k // 32))).astype(np.float16)[..., None].view(np.uint8)
    return b.reshape(n, -1)


def _decoder(gdev, seed=0, **kw):
    hp = dict(BASE, **kw)
    rng = np.random.default_rng(seed)
    dec = g.LlamaDecoder(gdev, **hp)
    e, f, v, c = hp["n_embd"], hp["n_ff"], hp["n_vocab"], hp["n_ctx"]
    dec.tensor("tok_embd").write(_q4(rng, v, e))
    dec.tensor("output").write(_q4(rng, v, e))
    dec.tensor("out_norm").write((1 + 0.1 * rng.standard_normal(e)).astype(np.float32))
    shapes = {"wq": (e, e), "wk": (e, e), "wv": (e, e), "wo": (e, e), "w_gate": (f, e), "w_up": (f, e), "w_down": (e, f)}
    ct = np.float16 if hp.get("kv_f16") else np.float32
    for i in range(hp["n_layer"]):
        for name, (n, k) in shapes.items():
            dec.tensor(name, i).write(_q4(rng, n, k))
        for name in ("attn_norm", "ffn_norm"):
            dec.tensor(name, i).write((1 + 0.1 * rng.standard_normal(e)).astype(np.float32))
        for name in ("k_cache", "v_cache"):
            dec.tensor(name, i).write(rng.standard_normal((c, e), dtype=np.float32).astype(ct))
    return dec, hp


def _rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return np.linalg.norm(a - b) / np.linalg.norm(b)


def _row(dec, hp, name, layer, n_past):
    t = dec.tensor(name, layer).to_cpu_tensor()
    if hp.get("kv_head_major"):
        return t.reshape(hp["n_head"], hp["n_ctx"], -1)[:, n_past]
    return t.reshape(hp["n_ctx"], -1)[n_past]


@pytest.mark.parametrize("kw, positions", [
    (dict(), (0, 1, 126, 127, 128, 159)),                                        # f32: one split of 128 keys, two
    (dict(kv_f16=True, n_ctx=530), (0, 254, 255, 256, 511, 512, 529)),           # f16: 256 keys a split
    (dict(kv_head_major=True, n_ctx=300), (5, 299)),
    (dict(n_ff=64, n_vocab=1), (3,)),                                            # the smallest: one slot in down
    (dict(n_embd=1664, n_head=13, n_ff=4096, n_vocab=48), (130,)),               # 35 workgroups of 48 rows: 16 over; one chunk
    (dict(n_embd=1024, n_head=8, n_ff=4160, n_vocab=49), (40,)),                 # two chunks, one slot in the second
    (dict(n_embd=640, n_head=5, n_ff=8256, n_vocab=2000), (60,)),                # three chunks, one slot in the third
    (dict(n_embd=4096, n_head=32, n_ff=12288, n_layer=1), (100,)),               # the widest
    (dict(n_layer=41), (17,)),                                                   # 41 layers: two launches
    (dict(n_ctx=8300), (8190, 8191, 8192)),                                      # 64 splits of keys; beyond: layer by layer
    (dict(n_embd=384, n_head=3), (60,)),                                         # narrower than 512: layer by layer
    (dict(n_embd=4224, n_head=33, n_ff=512, n_layer=1), (9,)),                   # wider: layer by layer
])
def test_step_equals_the_launches_it_replaces(gdev, kw, positions):
    print(kw, flush=True)
    dec, hp = _decoder(gdev, **kw)
    tol = TOL[bool(kw.get("kv_f16"))]
    for n_past in positions:
        got = {}
        for plan in (4, 5):
            dec.decode(7 % hp["n_vocab"], n_past, plan)
            got[plan] = [dec.logits().copy()] + [_row(dec, hp, n, i, n_past) for i in (0, hp["n_layer"] - 1) for n in ("k_cache", "v_cache")]
            assert dec.ops_per_step() == (2 + 4 * hp["n_layer"] if plan == 5 else 2 + 5 * hp["n_layer"])
        for a, b in zip(got[5], got[4]):
            assert np.all(np.isfinite(a)) and _rel(a, b) < tol, (n_past, _rel(a, b))
    dec.close()


@pytest.mark.parametrize("kw, n_past, grid", [
    (dict(), 0, True), (dict(), 159, True), (dict(kv_f16=True, kv_head_major=True), 30, True), (dict(n_ff=64, n_vocab=1), 3, True),
    (dict(n_embd=4096, n_head=32, n_ff=12288, n_layer=1), 100, True), (dict(n_layer=41), 17, True),
    (dict(n_ctx=8300), 8191, True), (dict(n_ctx=8300), 8192, False),               # 64 splits of 128 f32 keys, 65
    (dict(n_ctx=8300, kv_f16=True), 8299, True),
    (dict(n_embd=384, n_head=3), 60, False),                                       # narrower than 512
    (dict(n_embd=4224, n_head=33, n_layer=1), 9, False),                           # wider than 4096
    (dict(n_layer=251, n_embd=512, n_ff=64, n_vocab=8, n_ctx=4), 1, False)])
def test_which_steps_go_out_in_one_grid(gdev, kw, n_past, grid):
    dec, hp = _decoder(gdev, **kw)
    dec.decode(0, n_past, 4)
    assert dec.calls_per_step() == dec.ops_per_step() == 2 + 5 * hp["n_layer"]
    dec.decode(0, n_past, 5)
    assert dec.calls_per_step() == (1 if grid else 2 + 4 * hp["n_layer"])
    gdev.set_option(4, 2)      # a form of q | k | v and attention is asked for: layer by layer
    try:
        dec.decode(0, n_past, 5)
    finally:
        gdev.set_option(4, 0)
    assert dec.calls_per_step() == 2 + 4 * hp["n_layer"]
    dec.capture(0, n_past, 5)
    assert dec.calls_per_step() == (1 if grid else 2 + 4 * hp["n_layer"])
    dec.close()


def test_steps_repeat_recorded_and_interleaved(gdev):
    """The same bits every time: eager, from a graph with other steps between the replays, and beside another decoder of
    other sizes in the same context."""
    dec, hp = _decoder(gdev, n_embd=1024, n_head=8, n_ff=2816, n_vocab=4000, n_layer=4, n_ctx=400)
    other, _ = _decoder(gdev, seed=1, kv_f16=True, n_ctx=600)
    dec.decode(9, 300, 5)
    want = dec.logits().copy()
    other.decode(3, 590, 5)
    want_other = other.logits().copy()
    for _ in range(50):
        dec.decode(9, 300, 5)
        assert np.array_equal(dec.logits(), want)
    dec.capture(9, 300, 5)
    for i in range(5):
        dec.replay()
        assert np.array_equal(dec.logits(), want), i
        other.decode(3, 590, 5)
        assert np.array_equal(other.logits(), want_other), i
        dec.decode(10 + i, 301 + i, 5)
        assert not np.array_equal(dec.logits(), want)
        dec.decode(9, 300, (4, 5)[i % 2])     # the recorded step reads token and position from the device
    other.close()
    dec.close()


def test_two_contexts_on_two_threads():
    """Steps of two contexts at once on one device: the workgroups of each wait only for their own, of lower index, so neither
    keeps the other from finishing; the bits are those of a step alone."""
    import threading
    hp = dict(n_embd=2048, n_head=16, n_ff=5632, n_vocab=8000, n_layer=3, n_ctx=700)
    devs = [g.Device.gpu(0) for _ in range(2)]
    decs = [_decoder(d, seed=2 + i, kv_f16=bool(i), **hp)[0] for i, d in enumerate(devs)]
    want, bad = [], []
    for i, dec in enumerate(decs):
        dec.decode(5 + i, 600 + i, 5)
        want.append(dec.logits().copy())

    def work(i):
        try:
            for _ in range(150):
                decs[i].decode(5 + i, 600 + i, 5)
                if not np.array_equal(decs[i].logits(), want[i]):
                    bad.append(i)
        except g.GError as e:
            bad.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad[:3]
    for dec in decs:
        dec.close()


def test_bad_arguments_are_refused_and_leave_the_decoder_usable(gdev):
    dec, hp = _decoder(gdev)
    dec.decode(9, 20, 5)
    want = dec.logits().copy()
    for token, n_past in ((-1, 20), (hp["n_vocab"], 20), (9, -1), (9, hp["n_ctx"])):
        with pytest.raises(g.GError):
            dec.decode(token, n_past, 5)
    dec.decode(9, 20, 5)
    assert np.array_equal(dec.logits(), want)
    dec.close()


def test_waits_that_run_out_are_reported_once(gdev):
    """Every stage is made to wait for a tag that no element will carry, a few polls long: all waits run out, every
    workgroup still ends, the logits are NaN, the status comes once, and the next step is the one it was."""
    dec, _ = _decoder(gdev)
    dec.decode(9, 20, 5)
    want = dec.logits().copy()
    gdev.set_option(2, 64)
    gdev.set_option(3, 1)
    try:
        dec.decode(9, 20, 5)
        with pytest.raises(g.GError, match="-7"):
            dec.logits()
        assert np.all(np.isnan(dec.logits()))
    finally:
        gdev.set_option(2, 0)
        gdev.set_option(3, 0)
    dec.decode(9, 20, 5)
    assert np.array_equal(dec.logits(), want)
    dec.close()
