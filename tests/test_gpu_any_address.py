"""GPU parity of rows that start at any multiple of four bytes and are any number of logits long: the last group of one to three,
rows shorter than a group, what lies between the rows, mask bits behind a row's end, the count above a close token."""
import numpy as np
import pytest

from mako_amd import api, hip
from parity import oracle_rows

pytestmark = pytest.mark.gpu


def _kinds():
    p = api.make_params(7, 0.8)
    p["temperature"][0] = 0.0
    p["top_k"][1], p["top_p"][1] = 40, 0.9
    p["top_p"][2] = 0.9
    p["top_p"][3], p["min_p"][3] = 0.99, 0.01
    p["top_k"][5] = 3
    p["top_k"][6], p["top_p"][6] = 200, 0.9
    return p


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("vocab", [1, 2, 3, 4, 5, 7, 1022, 4095, 4097, 16383, 16385, 16387, 32770, 65537])
def test_rows_at_any_address(vocab, masked):
    rng = np.random.Generator(np.random.PCG64([vocab, masked]))
    p = _kinds()
    rows = len(p)
    hist_len = 60
    for name, v in (("repetition_penalty", 1.2), ("frequency_penalty", 0.2), ("presence_penalty", 0.3)):
        p[name][1:] = np.float32(v)
    w = dict(params=p, u=rng.random(rows).astype(np.float32))
    w["logits"] = (rng.standard_normal((rows, vocab)) * 2.0).astype(np.float32)
    w["hist"] = rng.integers(max(0, vocab - 40), vocab, (rows, hist_len)).astype(np.int32)  # (the row's end above all)
    w["hist_len"] = np.full(rows, hist_len, np.uint32)
    if masked:
        words = (vocab + 31) // 32
        w["mask"] = rng.integers(0, 2**32, (rows, words), dtype=np.uint64).astype(np.uint32)
        if vocab % 32:
            w["mask"][:, -1] |= np.uint32((0xFFFFFFFF << (vocab % 32)) & 0xFFFFFFFF)  # (no tokens there: nobody may look)
        w["mask"][:, 0] |= 1
    ref = oracle_rows(w)
    close = rng.integers(0, vocab, rows).astype(np.int32)
    allowed = np.ones((rows, vocab), bool)
    if masked:
        allowed = ((w["mask"][:, np.arange(vocab) >> 5] >> (np.arange(vocab, dtype=np.uint32) & 31)) & 1).astype(bool)
    above = ((w["logits"] > w["logits"][np.arange(rows), close][:, None]) & allowed).sum(1)
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab, max_hist=hist_len)
    try:
        for pad, offset in ((0, 0), (1, 0), (0, 1), (2, 3), (3, 2), (4, 4)):
            flat = np.full(offset + rows * (vocab + pad) - pad, 1e30, np.float32)  # (the last row ends with the allocation)
            for r in range(rows):
                flat[offset + r * (vocab + pad):][:vocab] = w["logits"][r]
            buf = hip.DeviceArray.from_host(flat)
            for hinted in (False, True):
                for closing in (False, True):
                    b = api.Batch(w["logits"], p, w["u"], mask=w.get("mask"), hist=w["hist"], hist_len=w["hist_len"], params_host=hinted,
                                  **(dict(close_token=close, close_max_above=0) if closing else {}))
                    b.desc.logits, b.desc.logits_stride = buf.ptr + 4 * offset, vocab + pad
                    ctx.sample_batch(b.desc, params_host=b.params_host)
                    g = b.results()
                    for r, (t, tr) in enumerate(ref):
                        what = (vocab, pad, offset, hinted, closing, r)
                        if closing and allowed[r, close[r]]:
                            assert g["above"][r] == above[r], what
                            if g["forced"][r] != api.FORCED_NONE:
                                continue
                        assert g["tokens"][r] == t, what
                        if p["temperature"][r] > 0:
                            assert g["n_cand"][r] == tr["n_cand"], what
                            assert np.float32(g["total"][r]).view(np.uint32) == np.float32(tr["total"]).view(np.uint32), what
    finally:
        ctx.close()
