"""GPU parity of rows that the whole-row path takes from their logits on (whole_row.h, copy_masked_row()): rows of equal logits,
whose candidate lists overflow, and rows in token order whose candidates are written out from a list with gaps; of lengths around
its trips and groups, at any address, with masks, histories and NaN."""
import numpy as np
import pytest

from mako_amd import api
from parity import assert_parity

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [1, 2, 3, 4, 5, 7, 514, 4095, 16383, 16384, 16385, 32771, 129281])
def test_whole_row_copy(vocab):
    rows = 6
    rng = np.random.Generator(np.random.PCG64(vocab))
    x = np.full((rows, vocab), 0.75, np.float32)
    x[:, vocab // 2] = 1.0
    x[2, ::3] = np.nan
    p = api.make_params(rows, 0.8, 40, 0.95)
    p["top_k"][3:5], p["top_p"][3:5] = 0, 1.0
    p["temperature"][5] = 0.0
    w = dict(name="copy V=%d" % vocab, logits=x, params=p, u=rng.random(rows).astype(np.float32))
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab, max_hist=32)
    try:
        for masked in (False, True):
            if masked:
                w["mask"] = rng.integers(0, 2**32, (rows, (vocab + 31) // 32), dtype=np.uint64).astype(np.uint32)
                w["mask"][1] = 0
                w["mask"][1, (vocab - 1) // 32] = 1 << ((vocab - 1) % 32)
                w["mask"][4] = 0xFFFFFFFF
                w["hist"] = rng.integers(0, vocab, (rows, 20)).astype(np.int32)
                w["hist_len"] = np.full(rows, 20, np.uint32)
                for name, v in (("repetition_penalty", 1.3), ("frequency_penalty", 0.2), ("presence_penalty", 0.3)):
                    p[name] = np.float32(v)
            for hinted in (True, False):
                g = assert_parity(ctx, w, cap=32, hinted=hinted)
                if vocab > 512 and not masked:
                    assert (g["path"][[0, 1]] == api.PATH_GENERAL).all(), g["path"]
    finally:
        ctx.close()
