"""GPU parity of rows in token order that few of their logits are candidates of (index_rows.h, few_candidates_row()): up to the
256 that a list of their own may hold and beyond, in one piece of 16 384 logits or in all of them, at the pieces' edges, drawn,
verified and scored, in launches of their own and beside other rows."""
import numpy as np
import pytest

from mako_amd import api
from parity import gpu_rows, oracle_rows

pytestmark = pytest.mark.gpu


def _batch(vocab, seed):
    rng = np.random.Generator(np.random.PCG64([seed, vocab]))
    counts = [c for c in (1, 2, 63, 64, 65, 255, 256, 257, 300) if c <= vocab]
    rows = 2 * len(counts)
    x = np.full((rows, vocab), -np.inf, np.float32)
    edges = [i for i in (0, 255, 256, 4095, 4096, 16383, 16384, 32767, 32768, vocab - 1) if i < vocab]
    for r in range(rows):
        n = counts[r // 2]
        span = vocab if r % 2 else min(vocab, max(n, 300))  # (anywhere, or in a stretch)
        first = rng.integers(0, vocab - span + 1)
        at = np.concatenate([rng.permutation(edges)[: n // 2] if r % 2 else [], first + rng.permutation(span)]).astype(np.int64)
        at = at[np.sort(np.unique(at, return_index=True)[1])][:n]
        x[r, at] = rng.standard_normal(n) * 0.5
    p = api.make_params(rows, 0.8, 0, 1.0)
    p["min_p"][::3] = np.float32(0.05)
    u = np.resize(np.float32([0.0, 2.0**-24, 0.3, 0.7, 0.999, 1.0 - 2.0**-24]), rows)
    rng.shuffle(u)
    return dict(name="few, V=%d" % vocab, logits=x, params=p, u=u), rng


@pytest.mark.parametrize("vocab", [1, 2, 257, 4097, 16384, 16385, 40000, 151553, 262144])
def test_few_candidates(vocab):
    w, rng = _batch(vocab, 1)
    rows = len(w["u"])
    draft = np.array([rng.choice(np.flatnonzero(np.isfinite(w["logits"][r]))) if r % 3 else rng.integers(vocab) for r in range(rows)], np.int32)
    u2 = rng.random(rows).astype(np.float32)
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)
    try:
        for beside in (False, True):
            if beside and vocab > 2:
                w["params"]["top_p"][0], w["params"]["top_k"][1] = 0.9, 30
            ref, verified = oracle_rows(w), oracle_rows(w, draft=draft, u2=u2)
            for hinted in (True, False):
                g, v = gpu_rows(ctx, w, hinted=hinted), gpu_rows(ctx, w, draft=draft, u2=u2, hinted=hinted)
                for r in range(rows):
                    t, tr = ref[r]
                    assert (g["tokens"][r], g["n_cand"][r]) == (t, tr["n_cand"]), (r, hinted)
                    assert np.float32(g["total"][r]).view(np.uint32) == np.float32(tr["total"]).view(np.uint32), (r, hinted)
                    assert np.float32(g["q"][r]).view(np.uint32) == np.float32(tr["q_chosen"]).view(np.uint32), (r, hinted)
                    assert (v["tokens"][r], bool(v["accepted"][r])) == (verified[r][0], bool(verified[r][1]["accepted"])), (r, hinted)
    finally:
        ctx.close()


# (rows of a few groups of 256, for which records would be as short as the list)
@pytest.mark.parametrize("vocab", [2, 255, 256, 257, 512, 513, 640, 641, 20000])
def test_few_candidates_of_short_rows(vocab):
    rng = np.random.Generator(np.random.PCG64([9, vocab]))
    ends = [e for e in (1, 255, 256, 257, 511, 512, 513, vocab) if e <= vocab]
    counts = [c for c in (1, 2, 100, 255, 256, 257, 500) if c <= vocab]
    x = np.full((len(ends) * len(counts), vocab), -np.inf, np.float32)
    for r, (end, n) in enumerate((e, c) for e in ends for c in counts):
        at = np.append(rng.permutation(end - 1)[: n - 1], end - 1)
        x[r, at] = rng.standard_normal(len(at)) * 0.5
    rows = len(x)
    p = api.make_params(rows, 0.8, 0, 1.0)
    u = np.resize(np.float32([0.0, 0.3, 0.7, 1.0 - 2.0**-24]), rows)
    w = dict(name="few, short, V=%d" % vocab, logits=x, params=p, u=u)
    draft, u2 = np.argmax(x, 1).astype(np.int32), rng.random(rows).astype(np.float32)
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)
    try:
        ref, verified = oracle_rows(w), oracle_rows(w, draft=draft, u2=u2)
        for hinted in (True, False):
            g, v = gpu_rows(ctx, w, hinted=hinted), gpu_rows(ctx, w, draft=draft, u2=u2, hinted=hinted)
            for r in range(rows):
                t, tr = ref[r]
                assert (g["tokens"][r], g["n_cand"][r]) == (t, tr["n_cand"]), (r, hinted)
                assert np.float32(g["total"][r]).view(np.uint32) == np.float32(tr["total"]).view(np.uint32), (r, hinted)
                assert (v["tokens"][r], bool(v["accepted"][r])) == (verified[r][0], bool(verified[r][1]["accepted"])), (r, hinted)
    finally:
        ctx.close()
