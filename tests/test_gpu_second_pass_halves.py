"""GPU parity of the second pass's workgroups of 512 threads (large batches): vocabularies around their pieces of 8 192 logits and
the blocks of 2 048 that those are cut into, rows at any address, and histories that take none, two or four entries a thread, or the
workgroups of 1 024."""
import numpy as np
import pytest

from mako_amd import api
from parity import assert_parity, nucleus_batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hist", [0, 1, 1024, 1025, 2048, 2049])
@pytest.mark.parametrize("vocab", [2047, 2048, 6145, 8192, 8193, 16384, 24577, 61440, 65537, 114689])
def test_pieces(vocab, hist):
    rows = 40
    w = nucleus_batch(rows, vocab, vocab + hist, [0.05, 0.6, 2.5, 5.0], [1.0, 0.7], [0.9, 0.999], us=[0.0, 0.3, 0.98])
    if hist:
        rng = np.random.Generator(np.random.PCG64([vocab, hist]))
        p = w["params"]
        p["repetition_penalty"], p["frequency_penalty"], p["presence_penalty"] = 1.1, 0.2, 0.3
        w["hist"] = rng.integers(0, vocab, (rows, hist)).astype(np.int32)
        w["hist"][:, : hist // 2] //= 64 # (half of them among the first tokens)
        w["hist_len"] = rng.integers(0, hist + 1, rows).astype(np.uint32)
        w["hist_len"][:4] = hist
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab, max_hist=max(hist, 1))
    try:
        assert_parity(ctx, w, cap=64, hinted=True)
    finally:
        ctx.close()


@pytest.mark.parametrize("rows", [65, 129, 257])
def test_workgroups_of_several_pieces(rows):
    vocab = 40000
    w = nucleus_batch(rows, vocab, rows, [0.05, 0.6, 2.5, 5.0], [1.0, 0.7], [0.9, 0.999], us=[0.0, 0.3, 0.98])
    w["params"]["top_k"][3::7] = 40
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)
    try:
        for hinted in (True, False):
            assert_parity(ctx, w, cap=64, hinted=hinted)
    finally:
        ctx.close()
