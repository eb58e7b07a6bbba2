"""The launches of a batch of rows that take nth_element's rounds: as many for its steps as the rows' top_k leaves work for (counted
as the nodes of a captured graph, which is not run)."""
import ctypes

import numpy as np
import pytest

from mako_amd import api, hip

pytestmark = pytest.mark.gpu


def _launches(ctx, vocab, params):
    lib, rows = hip.lib(), len(params)
    x = np.random.Generator(np.random.PCG64(vocab)).standard_normal((rows, vocab)).astype(np.float32)
    b = api.Batch(x, params, np.full(rows, 0.5, np.float32), params_host=True)
    ctx.sample_batch(b.desc, params_host=b.params_host)  # (what a first call sets up)
    hip.synchronize()
    stream, graph, nodes = hip.Stream(), ctypes.c_void_p(), ctypes.c_size_t()
    hip.check(lib.hipStreamBeginCapture(ctypes.c_void_p(stream.ptr), 2), "hipStreamBeginCapture")
    try:
        ctx.sample_batch(b.desc, stream=stream, params_host=b.params_host)
    finally:
        hip.check(lib.hipStreamEndCapture(ctypes.c_void_p(stream.ptr), ctypes.byref(graph)), "hipStreamEndCapture")
    hip.check(lib.hipGraphGetNodes(graph, None, ctypes.byref(nodes)), "hipGraphGetNodes")
    hip.check(lib.hipGraphDestroy(graph), "hipGraphDestroy")
    return nodes.value


# (the other launches: scan, weights and tail, and the groups of rows in token order)
@pytest.mark.parametrize("vocab, top_ks, top_p, others, steps", [
    (129280, (40, 40), 1.0, 3, 4), (129280, (129280, 2**32 - 1), 1.0, 3, 1), (129280, (60000,), 1.0, 3, 1), (129280, (13000,), 1.0, 3, 2),
    (129280, (60000, 40), 1.0, 3, 4), (129280, (500, 900), 0.9, 3, 1), (129280, (0, 500), (1.0, 0.9), 4, 1), (129280, (0, 0), 1.0, 4, 0),
    (129280, (60000, 500), (1.0, 0.9), 3, 1), (40000, (40,), 1.0, 3, 2), (40000, (39999,), 1.0, 3, 1), (32768, (40,), 1.0, 3, 0),
])
def test_launches(vocab, top_ks, top_p, others, steps):
    p = api.make_params(len(top_ks), 0.8, 0, 1.0)
    p["top_k"] = top_ks
    p["top_p"] = np.float32(top_p)
    ctx = api.SamplerContext(max_rows=len(top_ks), max_vocab=vocab)
    try:
        assert _launches(ctx, vocab, p) == others + steps
    finally:
        ctx.close()
