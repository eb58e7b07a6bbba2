"""GPU parity of rows of few logits per wave that are too long for a candidate list of all of them (513 to 5 116): top-k rows of any
such length are finished from their candidates, aligned or not, whatever their histories penalise."""
import numpy as np
import pytest

from mako_amd import api
from parity import assert_parity

pytestmark = pytest.mark.gpu


def _batch(vocab, seed):
    rng = np.random.Generator(np.random.PCG64([seed, vocab]))
    top_ks = [1, 2, 20, 40, 50, 100, 128, 0, 0, 0, 0]
    rows = len(top_ks)
    x = (rng.standard_normal((rows, vocab)) * 3.0).astype(np.float32)
    x[8] *= np.float32(0.02)
    x[9, :50] += np.float32(10.0)
    p = api.make_params(rows, 0.8, 0, 0.95)
    p["top_k"] = top_ks
    p["top_p"][10] = np.float32(0.5)
    return dict(name="short V=%d" % vocab, logits=x, params=p, u=rng.random(rows).astype(np.float32))


# (512: the longest row whose list may hold all of it; around whole groups of 256, and of 4 096; 5 116: the longest
# of these rows)
@pytest.mark.parametrize("vocab", [511, 512, 513, 600, 681, 767, 768, 769, 1003, 2048, 2049, 3001, 3840, 3841, 3845, 3899, 4092, 4093, 4096, 4097, 5115, 5116, 5117, 5121])
def test_short_rows(vocab):
    w = _batch(vocab, 1)
    ctx = api.SamplerContext(max_rows=16, max_vocab=vocab, max_hist=64)
    try:
        for hinted in (True, False):
            g = assert_parity(ctx, w, cap=600, hinted=hinted)
            assert (g["path"][:6] == api.PATH_TOPK).all(), g["path"]
        # with what makes logits equal, missing and moved
        w["logits"][1::2] = np.round(w["logits"][1::2])
        w["logits"][:, 256:300] = -np.inf
        w["logits"][3, ::7] = np.nan
        rng = np.random.Generator(np.random.PCG64(vocab))
        w["mask"] = rng.integers(0, 2**32, (len(w["u"]), (vocab + 31) // 32), dtype=np.uint64).astype(np.uint32)
        w["mask"][0] = 0xFFFFFFFF
        for name, v in (("repetition_penalty", 1.3), ("frequency_penalty", 0.2), ("presence_penalty", 0.3)):
            w["params"][name] = np.float32(v)
        w["hist"] = rng.integers(0, vocab, (len(w["u"]), 50)).astype(np.int32)
        w["hist_len"] = np.full(len(w["u"]), 50, np.uint32)
        for hinted in (True, False):
            assert_parity(ctx, w, cap=600, hinted=hinted)
    finally:
        ctx.close()


# (a history that names the first tokens most often, on rows as flat as they come: those tokens' logits are no one's candidates)
@pytest.mark.parametrize("vocab", [600, 901, 2067, 2068, 3068, 4101, 4352, 5116])
@pytest.mark.parametrize("hist", [1000, 2048, 5000, 9000])
def test_short_rows_with_long_histories(vocab, hist):
    rows = 5
    rng = np.random.Generator(np.random.PCG64([vocab, hist]))
    p = api.make_params(rows, 0.7, 40, 0.95)
    p["top_k"][1], p["top_k"][4], p["top_p"][4] = 20, 0, 0.9
    for name, v in (("repetition_penalty", 1.1), ("frequency_penalty", 0.2), ("presence_penalty", 0.3)):
        p[name] = np.float32(v)
    cdf = np.cumsum(np.arange(1, vocab + 1) ** -1.1)
    w = dict(name="V=%d hist=%d" % (vocab, hist), params=p, logits=(rng.standard_normal((rows, vocab)) * 0.1).astype(np.float32),
             u=rng.random(rows).astype(np.float32), hist_len=np.full(rows, hist, np.uint32),
             hist=np.minimum(np.searchsorted(cdf, rng.random((rows, hist)) * cdf[-1]), vocab - 1).astype(np.int32))
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab, max_hist=hist)
    try:
        for hinted in (True, False):
            g = assert_parity(ctx, w, cap=600, hinted=hinted)
            assert (g["path"][:4] == api.PATH_TOPK).all(), g["path"]
    finally:
        ctx.close()
