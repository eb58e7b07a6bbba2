"""GPU parity of batches whose rows of the whole-row class are finished in the launches of the others' kernels: every kind of
row beside every other, with and without the caller's host copy of the parameters, over more rows than a wave has lanes, with
vocabularies whose logits are loaded one at a time, masks and forced rows among them."""
import numpy as np
import pytest

from mako_amd import api, workloads
from parity import assert_parity, gpu_rows

pytestmark = pytest.mark.gpu


def _batch(rows, vocab, kinds, seed):
    rng = np.random.Generator(np.random.PCG64([seed, rows, vocab]))
    logits = (rng.standard_normal((rows, vocab)) * 3.0).astype(np.float32)
    p = api.make_params(rows, 0.9, 0, 1.0)
    kind = np.array(kinds)[rng.permutation(np.arange(rows) % len(kinds))]
    p["temperature"][kind == "greedy"] = 0.0
    p["top_k"][kind == "top_k"], p["top_p"][kind == "top_k"] = 40, np.float32(0.95)
    p["top_p"][kind == "nucleus"] = np.float32(0.97)
    p["min_p"][kind == "min_p"] = np.float32(0.05)
    p["top_k"][kind == "top_k_alone"] = 30
    p["top_k"][kind == "wide_top_k"], p["top_p"][kind == "wide_top_k"] = 500, np.float32(0.9)
    w = dict(name="beside %d x %d" % (rows, vocab), logits=logits, params=p, u=workloads._uniforms(rng, rows))
    words = (vocab + 31) // 32
    bits = rng.random((rows, words * 32)) < 0.7
    bits[::2] = True
    bits[:, vocab:] = False
    w["mask"] = np.ascontiguousarray(np.packbits(bits.reshape(rows, words, 32), axis=2, bitorder="little").view(np.uint32).reshape(rows, words))
    return w


ALL = ["greedy", "top_k", "nucleus", "temperature", "min_p", "top_k_alone", "wide_top_k"]


@pytest.mark.parametrize("rows", [1, 7, 64, 65, 130])
@pytest.mark.parametrize("vocab", [4099, 16384, 33000])
@pytest.mark.parametrize("kinds", [ALL, ["top_k", "temperature"], ["greedy", "wide_top_k"], ["nucleus", "top_k_alone"]])
def test_every_kind_beside_every_other(rows, vocab, kinds):
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)
    try:
        w = _batch(rows, vocab, kinds, 5)
        a = assert_parity(ctx, w, cap=0, hinted=True)
        b = assert_parity(ctx, w, cap=0)
        c = gpu_rows(ctx, w, cap=64)
        assert np.array_equal(a["tokens"], b["tokens"]) and np.array_equal(a["tokens"], c["tokens"])
        assert np.array_equal(a["path"], b["path"])
    finally:
        ctx.close()


@pytest.mark.parametrize("kinds", [ALL, ["top_k"], ["nucleus", "temperature"]])
def test_more_pieces_than_workgroups(kinds):
    """Thousands of rows: a workgroup beside the others' takes dozens of pieces in turn and looks for each one's row."""
    rows, vocab = 5003, 300
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)
    try:
        w = _batch(rows, vocab, kinds, 9)
        a = assert_parity(ctx, w, cap=8)
        b = gpu_rows(ctx, w, hinted=True)
        assert np.array_equal(a["tokens"], b["tokens"])
    finally:
        ctx.close()
