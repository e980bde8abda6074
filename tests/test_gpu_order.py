"""Launches whose workgroups wait for one another, sent out by two contexts on one device: the one that comes second runs behind
the first (directly, from a graph, and in the launch of q | k | v and attention), whatever its own stream has left; a context that
is capturing or gone holds nobody up."""
import numpy as np
import pytest

from galois_amd import Device
from tests.test_gpu_llama_step_abi import V, _Model

pytestmark = pytest.mark.gpu


class _Side:
    def __init__(self, seed):
        self.dev = Device(0)
        self.model, self.ev = _Model(self.dev, seed), self.dev.event()
        self.n = 1 << 26
        self.x = self.dev.alloc(self.n * 4)
        self.want = self.step_now()
        # q | k | v and the attention in one launch, on vectors of their own
        m = self.model.m
        self.bufs = [self.dev.upload(np.linspace(-1, 1, m.n_embd, dtype=np.float32)) for _ in range(5)]
        y, (x, q, k, v, self.out) = self.model.layers[0], self.bufs
        self.items = self.dev.gemv_items([dict(vx=w, y=x, dst=d, ncols=m.n_embd, nrows=m.n_embd) for w, d in ((y.wq, q), (y.wk, k), (y.wv, v))])

    def busy(self):
        """Some ten milliseconds of other work on this context's stream."""
        for _ in range(60):
            self.dev.scale_f32(self.x, self.x, 1.0, self.n)

    def step(self):
        assert self.model.step(7, 100) == 0

    def step_now(self):
        self.step()
        return self.model.get("logits", np.float32, V)

    def attention(self):
        m, y = self.model.m, self.model.layers[0]
        self.dev.set_option(Device.OPT_QKV_ATTN_LAUNCHES, 1)
        self.dev.qkv_attn_decode(self.items, y.k_cache, y.v_cache, self.out, m.n_head, 128, 100, m.pos, 1.0, m.theta_scale, m.scale)
        self.dev.set_option(Device.OPT_QKV_ATTN_LAUNCHES, 0)

    def close(self):
        self.dev.close()


@pytest.mark.parametrize("first", ["step", "attention", "graph"])
@pytest.mark.parametrize("second", ["step", "attention", "graph"])
def test_the_second_context_runs_behind_the_first(first, second):
    a, b = _Side(1), _Side(2)
    graphs = []
    for s in (a, b):
        s.dev.graph_begin_capture()
        s.step()
        graphs.append(s.dev.graph_end_capture())
    for _ in range(2):
        a.busy()
        a.dev.graph_launch(graphs[0]) if first == "graph" else getattr(a, first)()
        a.dev.record(a.ev)
        b.dev.graph_launch(graphs[1]) if second == "graph" else getattr(b, second)()
        b.dev.record(b.ev)
        a.dev.synchronize(), b.dev.synchronize()
        assert a.dev.elapsed_ms(a.ev, b.ev) >= 0.0   # without an order b is done while a's stream is still busy
        a, b, graphs = b, a, graphs[::-1]
        first, second = second, first
    for s in (a, b):
        assert np.array_equal(s.step_now(), s.want)
    for s, g in zip((a, b), graphs):
        s.dev.graph_destroy(g)
        s.close()


def test_contexts_that_capture_or_have_gone():
    a, b, c = _Side(3), _Side(4), _Side(5)
    logits = lambda s: s.model.get("logits", np.float32, V)
    a.step()
    a.dev.graph_begin_capture()      # a's launch is the device's last, and nothing can be recorded on its stream now
    a.step()
    b.step()
    c.step()
    b.step()
    g = a.dev.graph_end_capture()
    assert np.array_equal(logits(b), b.want) and np.array_equal(logits(c), c.want)
    for _ in range(3):
        a.dev.graph_launch(g)
        b.step()
        assert np.array_equal(logits(a), a.want)
        assert np.array_equal(a.step_now(), a.want) and np.array_equal(logits(b), b.want)
    a.dev.graph_destroy(g)
    a.step()
    a.close()
    b.step()
    c.step()
    assert np.array_equal(logits(b), b.want) and np.array_equal(logits(c), c.want)
    b.close(), c.close()
