"""GPU parity of std::ranges::nth_element's replay (src/gen/sampler.cpp:39-43) at the sizes where its ways of making a round
meet: ranges in device memory, in a workgroup's registers and in one wave's, and the sorts of the survivors before a top-p."""
import numpy as np
import pytest

from mako_amd import api
from parity import assert_parity

pytestmark = pytest.mark.gpu


def _batch(vocab, top_ks, top_p, seed, ties):
    rng = np.random.Generator(np.random.PCG64([seed, vocab]))
    rows = len(top_ks)
    logits = (rng.standard_normal((rows, vocab)) * 2.0).astype(np.float32)
    if ties:  # few different weights: equal ones are told apart by their token ids, also from the pivot
        logits = np.round(logits * 4.0) / np.float32(4.0)
    p = api.make_params(rows, 0.8, 0, top_p)
    p["top_k"] = top_ks
    return dict(name="nth_element V=%d" % vocab, logits=logits, params=p, u=rng.random(rows).astype(np.float32))


# (16 380 entries fit the registers wherever the range begins; 256 a wave; LDS has no room for the bits of more than 524 288)
@pytest.mark.parametrize("vocab", [3, 5, 255, 256, 257, 1025, 4097, 16379, 16380, 16381, 16384, 16385, 16640, 40001, 262144, 530001])
@pytest.mark.parametrize("ties", [False, True])
def test_top_k_alone(vocab, ties):
    top_ks = sorted({k for k in (1, 2, 3, 40, 255, 256, 257, 1000, vocab // 2, vocab - 1) if 0 < k < vocab})
    ctx = api.SamplerContext(max_rows=len(top_ks), max_vocab=vocab)
    try:
        w = _batch(vocab, top_ks, 1.0, 1, ties)
        for hinted in (True, False):
            assert_parity(ctx, w, cap=256, hinted=hinted)
    finally:
        ctx.close()


@pytest.mark.parametrize("top_k", [129, 256, 257, 1023, 1024, 1025, 4095, 4096, 4097, 9000])
def test_sorted_survivors(top_k):
    vocab = 20000
    ctx = api.SamplerContext(max_rows=4, max_vocab=vocab)
    try:
        for ties in (False, True):
            w = _batch(vocab, [top_k] * 4, 0.97, top_k, ties)
            for hinted in (True, False):
                assert_parity(ctx, w, cap=256, hinted=hinted)
    finally:
        ctx.close()
