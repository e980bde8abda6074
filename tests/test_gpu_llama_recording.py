"""A decode step inside a graph that the caller records on the decoder's context: one whose token and position are already on the
device is recorded, another is refused (it would change what later steps read, at times the decoder does not see), and either way the
next step computes its own token."""
import ctypes as C

import numpy as np
import pytest

from galois_amd import _abi
from galois_amd import host_api as g
from tests.test_gpu_llama_step import _decoder

pytestmark = pytest.mark.gpu


def _context(device):
    """The C ABI's context of an op-layer device: its first member points to an object whose first member it is."""
    return C.c_void_p.from_address(C.c_void_p.from_address(device.h).value)


@pytest.mark.parametrize("fused", [0, 4, 5])
def test_other_inputs_are_refused_while_the_caller_records(fused):
    gdev, lib = g.Device.gpu(0), _abi.load()
    ctx = _context(gdev)
    # 512 columns: plan 5 is the step in one grid, which stores token and position itself
    dec, hp = _decoder(gdev)
    dec.decode(7, 5, fused)
    want = np.array(dec.logits())
    dec.decode(3, 5, fused)
    assert lib.galois_hip_graph_begin_capture(ctx) == 0
    graph = C.c_void_p()
    try:
        for token, n_past in ((7, 5), (3, 6), (7, 6)):
            with pytest.raises(g.GError):
                dec.decode(token, n_past, fused)
        dec.decode(3, 5, fused)
    finally:
        assert lib.galois_hip_graph_end_capture(ctx, C.byref(graph)) == 0
    dec.decode(7, 5, fused)  # position 5 again: the same rows of the caches
    assert np.array_equal(dec.logits(), want)
    # the recorded step reads the token that is on the device
    assert lib.galois_hip_graph_launch(ctx, graph) == 0
    assert np.array_equal(dec.logits(), want)
    assert lib.galois_hip_graph_destroy(ctx, graph) == 0
    dec.close()
