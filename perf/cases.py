"""The workloads this library is measured on, each through the entry points a program calls.

A case is a dict of plain values; `listed()` names the fixed ones, `draw(rng)` makes another one of the same ranges.
`prepare(case, seed)` makes what a program holds before the call (a loaded model with its KV cache, weights and
activations on the device), `run(state)` is one pass, `work(case)` what the pass cannot do without, and
`tolerance(case)` how far two correct implementations at this precision may lie apart.

Kinds:
  decode    tokens one after the other through `LlamaDecoder.decode`, the logits fetched after each (as a sampler
            needs them)
  prefill   a prompt, or the next turn of a conversation, through `LlamaDecoder.prefill`, and its last token's logits
  gemv      Q4_0 matrix-vector products of one decode step, grouped into one call
  matmul    Q4_0 weights against a batch of f32 activation rows
  rows      the row operations around the products: norm, rotation, causal softmax
  quantize  f32 weights to Q4_0 and back, as a model is converted and checked
"""
import math

import numpy as np
import torch

import galois_amd
from galois_amd import host_api

QK = 32            # weights of a Q4_0 block
BLOCK_BYTES = 18   # bytes of a Q4_0 block
EPS = 1e-6
FREQ_BASE = 10000.0

_devices = {}


def _raw():
    """The C ABI's device (one context for the process, as a program keeps it)."""
    if "raw" not in _devices:
        _devices["raw"] = galois_amd.Device(0)
    return _devices["raw"]


def _host():
    """The op layer's device."""
    if "host" not in _devices:
        _devices["host"] = host_api.Device.gpu(0)
    return _devices["host"]


def _model(**kw):
    """The 32-layer model of the benchmark (d_model 4096, 32 heads of 128, FFN 11008, vocabulary 32000)."""
    return dict(dict(n_layer=32, n_embd=4096, n_head=32, n_ff=11008, n_vocab=32000), **kw)


def listed():
    return [
        # generation with a full context: the benchmark's decode step (KV length 2048, f32 caches), in the fastest
        # launch plan
        _model(name="decode_kv2048", kind="decode", n_past=2044, steps=4, kv="f32", plan=5),
        # the ordinary chat turn: a short context, caches in f16
        _model(name="decode_kv203_f16", kind="decode", n_past=200, steps=4, kv="f16", plan=5),
        # the default launch plan (one op per launch, as the ops of the reference are called) on a small model with
        # heads of 64: nothing but launches and latency
        dict(name="decode_ops_small", kind="decode", n_layer=8, n_embd=1024, n_head=16, n_ff=2816, n_vocab=32000, n_past=77,
             steps=2, kv="f32", plan=0),
        # the benchmark's prompt, a whole context in one pass, a one-sentence prompt
        _model(name="prefill_512", kind="prefill", n_past=0, tokens=512, kv="f32"),
        _model(name="prefill_2048", kind="prefill", n_past=0, tokens=2048, kv="f32"),
        _model(name="prefill_23", kind="prefill", n_past=0, tokens=23, kv="f32"),
        # the next question of a conversation that is already in the (f16) caches
        _model(name="prefill_150_past1201_f16", kind="prefill", n_past=1201, tokens=150, kv="f16"),
        # the benchmark's headline: the four matrix shapes of a decode step in one call
        dict(name="gemv_set", kind="gemv", products="4096x4096 4096x11008 11008x4096 4096x32000"),
        # the benchmark's prefill product on f32 activations
        dict(name="matmul_512x4096x11008", kind="matmul", m=512, k=4096, n=11008),
        # a model width that is no multiple of 256, a batch that is no multiple of anything
        dict(name="matmul_77x3200x8640", kind="matmul", m=77, k=3200, n=8640),
        # the benchmark's row operations: 512 tokens of a 4096-wide model with 32 heads
        dict(name="rows_512x4096", kind="rows", rows=512, n_embd=4096, n_head=32, n_past=0),
        # one feed-forward matrix converted
        dict(name="quantize_11008x4096", kind="quantize", n=11008, k=4096),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "prefill", "gemv", "matmul", "matmul", "rows", "quantize"])
    if kind in ("decode", "prefill"):
        d = 128 if rng.random() < 0.75 else 64
        e = 256 * rng.randint(4, 16)
        f = 256 * max(4, round(e * rng.uniform(2.5, 3.0) / 256))
        c = dict(kind=kind, n_layer=_log(rng, 4, 32), n_embd=e, n_head=e // d, n_ff=min(f, 11008), n_vocab=32000,
                 kv=rng.choice(["f32", "f16"]))
        if kind == "decode":
            plan = (5 if d == 128 else 4) if c["kv"] == "f16" or rng.random() < 0.75 else 0
            return dict(c, n_past=_log(rng, 1, 4000), steps=rng.randint(1, 4), plan=plan)
        n = _log(rng, 2, 1600)
        past = 0 if rng.random() < 0.6 else _log(rng, 16, 2000)
        if d == 64:  # the attention as single ops holds the scores of all heads
            n, past = min(n, 700), min(past, 700)
        return dict(c, n_past=past, tokens=n)
    if kind == "gemv":
        shapes = ["%dx%d" % (64 * _log(rng, 8, 172), _log(rng, 512, 32000)) for _ in range(rng.randint(1, 4))]
        return dict(kind="gemv", products=" ".join(shapes))
    if kind == "matmul":
        k = 256 * rng.randint(4, 43) if rng.random() < 0.6 else 32 * _log(rng, 16, 344)
        return dict(kind="matmul", m=_log(rng, 2, 1024), k=k, n=_log(rng, 512, 16000))
    if kind == "rows":
        return dict(kind="rows", rows=_log(rng, 8, 1024), n_embd=128 * rng.randint(8, 48), n_head=rng.randint(8, 40),
                    n_past=0 if rng.random() < 0.5 else _log(rng, 10, 1000))
    return dict(kind="quantize", n=_log(rng, 256, 32000), k=32 * _log(rng, 16, 344))


# ---- preparation -------------------------------------------------------------------------------------------------
class _Owner:
    """Frees a decoder with its memory when nothing refers to either any more."""

    def __init__(self, dec):
        self.dec = dec

    def __del__(self):
        torch.cuda.synchronize()
        self.dec.close()


class _Memory:
    """Device memory of the library; a tensor made of it keeps its owner alive."""

    def __init__(self, owner, ptr, shape, dtype):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": tuple(shape), "typestr": dtype, "version": 2}


def _tensor_at(owner, ptr, shape, dtype):
    return torch.as_tensor(_Memory(owner, ptr, shape, dtype), device="cuda")


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(gen, *shape, std=1.0, mean=0.0):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32).mul_(std).add_(mean)


def _q4_rows(gen, n, k):
    """[n][k] weights N(0, 0.02) as Q4_0 bytes, by the library's quantizer."""
    w = _normal(gen, n * k, std=0.02)
    out = torch.empty(n * k // QK * BLOCK_BYTES, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()  # the library works on a stream of its own
    dev = _raw()
    dev.quantize_row_q4_0(w.data_ptr(), out.data_ptr(), n * k)
    dev.synchronize()
    return out


def _model_with_cache(case, seed, positions):
    """A loaded model with random weights and a filled cache: its owner and the caches of its layers as tensors."""
    gen, dev = _generator(seed), _raw()
    e, f, v, c = case["n_embd"], case["n_ff"], case["n_vocab"], positions
    dec = host_api.LlamaDecoder(_host(), n_vocab=v, n_embd=e, n_head=case["n_head"], n_layer=case["n_layer"], n_ff=f, n_ctx=c,
                                rms_eps=EPS, freq_base=FREQ_BASE, kv_f16=case["kv"] == "f16")
    owner = _Owner(dec)
    stage = torch.empty(e * max(e, f, v), dtype=torch.float32, device="cuda")

    def fill_q4(name, layer, count):
        w = stage[:count].normal_(0.0, 0.02, generator=gen)
        torch.cuda.synchronize()
        dev.quantize_row_q4_0(w.data_ptr(), dec.tensor(name, layer).data_ptr(), count)
        dev.synchronize()

    def view(name, layer, shape, dtype="<f4"):
        return _tensor_at(owner, dec.tensor(name, layer).data_ptr(), shape, dtype)

    fill_q4("tok_embd", -1, e * v)
    fill_q4("output", -1, e * v)
    view("out_norm", -1, (e,)).normal_(1.0, 0.1, generator=gen)
    caches = []
    for i in range(case["n_layer"]):
        for name, count in (("wq", e * e), ("wk", e * e), ("wv", e * e), ("wo", e * e), ("w_gate", e * f), ("w_up", e * f),
                            ("w_down", e * f)):
            fill_q4(name, i, count)
        for name in ("attn_norm", "ffn_norm"):
            view(name, i, (e,)).normal_(1.0, 0.1, generator=gen)
        pair = [view(name, i, (c, e), "<f2" if case["kv"] == "f16" else "<f4") for name in ("k_cache", "v_cache")]
        if case["n_past"]:  # what earlier tokens left: N(0, 0.02) weights times unit-variance activations
            for t in pair:
                t[:case["n_past"]].normal_(0.0, 0.02 * e ** 0.5, generator=gen)
        caches.append(pair)
    torch.cuda.synchronize()
    return owner, caches


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind in ("decode", "prefill"):
        n = case["steps"] if kind == "decode" else case["tokens"]
        owner, caches = _model_with_cache(case, seed, case["n_past"] + n)
        # the rows a pass appends to the caches, of every layer above the first (the first layer's are products of the
        # embeddings alone, and enter everything above)
        rows = [t[case["n_past"]:] for pair in caches[1:] for t in pair]
        tokens = np.random.default_rng(seed).integers(0, case["n_vocab"], n, dtype=np.int32)
        state.update(owner=owner, tokens=tokens, rows=rows)
        return state
    gen, dev = _generator(seed), _raw()
    if kind == "gemv":
        items, vectors, keep = [], {}, []
        for shape in case["products"].split():
            k, n = (int(t) for t in shape.split("x"))
            if k not in vectors:
                vectors[k] = _normal(gen, k)
            w, y = _q4_rows(gen, n, k), torch.zeros(n, device="cuda")
            keep.append((w, y))
            items.append(dict(vx=w.data_ptr(), y=vectors[k].data_ptr(), dst=y.data_ptr(), ncols=k, nrows=n))
        state.update(items=dev.gemv_items(items), keep=keep, vectors=vectors, out=[y for _, y in keep])
    elif kind == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        state.update(w=_q4_rows(gen, n, k), x=_normal(gen, m, k), y=torch.zeros(m, n, device="cuda"))
    elif kind == "rows":
        r, e, h = case["rows"], case["n_embd"], case["n_head"]
        cols = case["n_past"] + r
        state.update(x=_normal(gen, r, e), w=_normal(gen, e, std=0.1, mean=1.0), q=_normal(gen, r, h * 128),
                     pos=torch.arange(case["n_past"], cols, dtype=torch.int32, device="cuda"),
                     s=_normal(gen, h * r, cols, std=3.0))
        state.update({"%s_out" % t: torch.zeros_like(state[t]) for t in ("x", "q", "s")})
    else:
        k, n = case["k"], case["n"]
        state.update(w=_normal(gen, n * k, std=0.02), q=torch.zeros(n * k // QK * BLOCK_BYTES, dtype=torch.uint8, device="cuda"),
                     back=torch.zeros(n * k, device="cuda"))
    torch.cuda.synchronize()
    return state


# ---- one pass ----------------------------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "decode":
        dec, logits = state["owner"].dec, np.empty((case["steps"], case["n_vocab"]), np.float32)
        for i, token in enumerate(state["tokens"]):
            dec.decode(int(token), case["n_past"] + i, case["plan"])
            logits[i] = dec.logits()
        return {"logits": logits, "cache_rows": state["rows"]}
    if kind == "prefill":
        dec = state["owner"].dec
        dec.prefill(state["tokens"], case["n_past"])
        return {"logits": dec.logits(), "cache_rows": state["rows"]}
    dev = _raw()
    if kind == "gemv":
        dev.dequantize_mul_mat_vec_q4_0_group(state["items"])
        return state["out"]
    if kind == "matmul":
        dev.mul_mat_q4_0_f32(state["w"].data_ptr(), state["x"].data_ptr(), state["y"].data_ptr(), case["k"], case["n"], case["m"])
        return state["y"]
    if kind == "rows":
        r, e, h, past = case["rows"], case["n_embd"], case["n_head"], case["n_past"]
        dev.rms_norm_mul_f32(state["x"].data_ptr(), state["w"].data_ptr(), state["x_out"].data_ptr(), e, r, EPS)
        dev.rope_f32(state["q"].data_ptr(), state["q_out"].data_ptr(), 128, r * h, state["pos"].data_ptr(), 1.0, h,
                     FREQ_BASE ** (-2.0 / 128))
        dev.soft_max_causal_f32(state["s"].data_ptr(), state["s_out"].data_ptr(), past + r, r, h * r, past)
        return [state["x_out"], state["q_out"], state["s_out"]]
    count = case["n"] * case["k"]
    dev.quantize_row_q4_0(state["w"].data_ptr(), state["q"].data_ptr(), count)
    dev.dequantize_row_q4_0(state["q"].data_ptr(), state["back"].data_ptr(), count)
    return [state["q"], state["back"]]


# ---- what a pass cannot do without -------------------------------------------------------------------------------
def _q4(n):
    return n // QK * BLOCK_BYTES


def work(case):
    kind = case["kind"]
    if kind in ("decode", "prefill"):
        e, f, v, layers = case["n_embd"], case["n_ff"], case["n_vocab"], case["n_layer"]
        weights, cache = 4 * e * e + 3 * e * f, 2 * e * (2 if case["kv"] == "f16" else 4)
        if kind == "decode":  # every token reads the weights and its cache rows
            keys = sum(case["n_past"] + i + 1 for i in range(case["steps"]))
            return {"bytes": case["steps"] * (layers * _q4(weights) + _q4(e * v)) + layers * cache * keys,
                    "flops": 2 * case["steps"] * (layers * weights + e * v) + 4 * e * layers * keys}
        n, past = case["tokens"], case["n_past"]
        keys = n * past + n * (n + 1) // 2
        return {"bytes": layers * (_q4(weights) + cache * (past + n)) + _q4(e * v) + n * _q4(e),
                "flops": 2 * n * layers * weights + 2 * e * v + 4 * e * layers * keys}
    if kind == "gemv":
        shapes = [tuple(int(t) for t in s.split("x")) for s in case["products"].split()]
        return {"bytes": sum(_q4(k * n) + 4 * n for k, n in shapes) + 4 * sum({k for k, _ in shapes}),
                "flops": sum(2 * k * n for k, n in shapes)}
    if kind == "matmul":
        m, k, n = case["m"], case["k"], case["n"]
        return {"bytes": _q4(k * n) + 4 * m * (k + n), "flops": 2 * m * k * n}
    if kind == "rows":
        r, e, h, past = case["rows"], case["n_embd"], case["n_head"], case["n_past"]
        seen = h * (r * past + r * (r + 1) // 2)  # scores under the mask: the others are not read
        return {"bytes": 4 * (2 * r * e + e) + 8 * r * h * 128 + 4 * (seen + h * r * (past + r)),
                "flops": 4 * r * e + 6 * r * h * 64 + 5 * seen}
    n = case["n"] * case["k"]
    return {"bytes": 4 * n + 2 * _q4(n) + 4 * n, "flops": 4 * n}


def tolerance(case):
    """About four times what was measured on the listed cases."""
    kind = case["kind"]
    if kind == "decode":
        # one launch plan against another (other orders of the f32 sums): 7.4e-5; caches in f16 also differ by single
        # roundings (1.9e-4, at most one unit of f16)
        return {"rel": 7e-4, "max": 4e-3} if case["kv"] == "f16" else {"rel": 3e-4, "max": 1.5e-3}
    if kind == "prefill":
        # fp16 operands through 32 layers, against the same tokens decoded one by one with activations of 18 bits: 6.1e-3
        return {"rel": 1.5e-2, "max": 0.1}
    if kind == "gemv":
        return {"rel": 1.6e-5, "max": 7e-5}  # against f64: 4.1e-6, activations rounded to 18 bits per block
    if kind == "matmul":
        return {"rel": 1.1e-3, "max": 6e-3}  # against f64: 2.7e-4, both operands rounded to fp16
    if kind == "rows":
        # the rotation's angles are rounded to f32, which grows with the position: 1.2e-5 up to position 511
        at = max(1.0, (case["n_past"] + case["rows"]) / 512)
        return {"rel": 5e-5 * at, "max": 8e-4 * at}
    return "exact"
