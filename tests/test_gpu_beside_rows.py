"""GPU parity of batches whose rows of the whole-row class are finished in the launches of the others' kernels: every kind of
row beside every other, with and without the caller's host copy of the parameters, over more rows than a wave has lanes, with
vocabularies whose logits are loaded one at a time, masks, histories, drafts and forced rows among them."""
import numpy as np
import pytest

from mako_amd import api, workloads
from parity import assert_parity, gpu_rows, oracle_rows

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


def _with_histories(w, seed):
    rng = np.random.Generator(np.random.PCG64([seed, 3]))
    rows, vocab = w["logits"].shape
    p = w["params"]
    p["repetition_penalty"], p["frequency_penalty"], p["presence_penalty"] = 1.1, 0.2, 0.3
    w["hist"] = rng.integers(0, vocab, (rows, 200)).astype(np.int32)
    w["hist_len"] = rng.integers(0, 198, rows).astype(np.uint32)
    return w


@pytest.mark.parametrize("rows,vocab", [(7, 4099), (65, 33000), (130, 16384)])
@pytest.mark.parametrize("hinted", [False, True])
def test_drafts_and_histories(rows, vocab, hinted):
    """Verification of every kind of row: drafts that are likely, unlikely and masked out, accepted and redrawn."""
    rng = np.random.Generator(np.random.PCG64([rows, vocab, 4]))
    w = _with_histories(_batch(rows, vocab, ALL, 6), 6)
    draft = w["logits"].argmax(axis=1).astype(np.int32)
    draft[::3] = rng.integers(0, vocab, len(draft[::3]))
    u2 = workloads._uniforms(rng, rows)
    u2[::5] = [0.0, 1.0 - 2.0**-24][rows % 2]
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab, max_hist=200)
    try:
        assert_parity(ctx, w, cap=0, hinted=hinted)
        g = gpu_rows(ctx, w, draft=draft, u2=u2, hinted=hinted)
        bad = [r for r, (t, tr) in enumerate(oracle_rows(w, draft=draft, u2=u2))
               if g["tokens"][r] != t or bool(g["accepted"][r]) != bool(tr["accepted"])]
        assert not bad, [(r, int(g["path"][r])) for r in bad[:8]]
    finally:
        ctx.close()


@pytest.mark.parametrize("rows,vocab", [(7, 4099), (65, 33000), (130, 16384)])
@pytest.mark.parametrize("hinted", [False, True])
def test_forced_rows_and_appended_histories(rows, vocab, hinted):
    """force_token and close_token on some rows of every kind, and the chosen token appended to the row's history: the
    launches that begin the rows of the whole-row class leave the forced ones alone, and the last one writes them.  Twice, the
    second time with the histories the first has left."""
    rng = np.random.Generator(np.random.PCG64([rows, vocab, 5]))
    w = _with_histories(_batch(rows, vocab, ALL, 7), 7)
    masked = np.where(np.unpackbits(w["mask"].view(np.uint8), axis=1, bitorder="little")[:, :vocab] != 0, w["logits"], -np.inf)
    order = np.argsort(-masked, axis=1, kind="stable")
    force, close = np.full(rows, -1, np.int32), np.full(rows, -1, np.int32)
    force[::4] = rng.integers(0, vocab, len(force[::4]))
    close[1::3], close[2::6] = order[1::3, 1], order[2::6, 30]
    # (counted on the logits the sampler is given: masked, not penalised)
    above = [int((masked[r] > masked[r, close[r]]).sum()) if close[r] >= 0 else 0xffffffff for r in range(rows)]
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab, max_hist=200)
    try:
        b = api.Batch(w["logits"], w["params"], w["u"], mask=w["mask"], hist=w["hist"], hist_len=w["hist_len"], force_token=force,
                      close_token=close, close_max_above=3, append_history=True, params_host=hinted)
        for _ in range(2):
            ref = oracle_rows(w)
            ctx.sample_batch(b.desc, params_host=b.params_host)
            g = b.results()
            taken = (close >= 0) & (np.array(above) < 3)
            want = np.where(force >= 0, force, np.where(taken, close, [t for t, _ in ref]))
            assert np.array_equal(g["tokens"], want), np.flatnonzero(g["tokens"] != want)[:8]
            assert np.array_equal(g["forced"] != api.FORCED_NONE, (force >= 0) | taken)
            assert np.array_equal(g["above"], np.array(above, np.uint32))
            hist, length = b.history()
            for r in range(rows):
                w["hist"][r, w["hist_len"][r]] = want[r]
            w["hist_len"] += 1
            assert np.array_equal(length, w["hist_len"]) and np.array_equal(hist, w["hist"])
    finally:
        ctx.close()
