"""GPU parity of batches of many top_k == 0 rows with the caller's host copy of the parameters and no row of the whole-row class among
them: the second pass and the sort then run in workgroups of 512 threads (without the host copy, up to 262 144 logits, they are
workgroups of 1 024 beside other rows' kernels).  Everything a row can come with: masks, drafts, histories as tokens and as counts,
forced and close tokens, rows at any address; narrow nuclei; vocabularies up to the longest of which the pass takes pieces of 8 192
logits and beyond; and the checked libraries, with sound plans and with rash ones."""
import numpy as np
import pytest

from mako_amd import api, hip, workloads
from parity import assert_parity, gpu_rows, nucleus_batch, oracle_rows, random_large_batch

pytestmark = pytest.mark.gpu

CHECKED = 1 << 31  # the checks are compiled in; every other bit is a failed one


def _batch(rows, vocab, seed, mask=True, hist=200):
    """Flat, middling and peaked nuclei, every seventh row a top-k; masks and histories."""
    rng = np.random.Generator(np.random.PCG64([seed, rows, vocab]))
    w = nucleus_batch(rows, vocab, seed, [0.05, 0.6, 2.5, 5.0], [1.0, 0.7], [0.9, 0.999], us=[0.0, 0.3, 0.98], name="%d x %d" % (rows, vocab))
    p = w["params"]
    p["top_k"][3::7], p["top_p"][3::7] = 40, np.float32(0.95)
    if hist:
        p["repetition_penalty"], p["frequency_penalty"], p["presence_penalty"] = 1.1, 0.2, 0.3
        w["hist"] = rng.integers(0, vocab, (rows, hist)).astype(np.int32)
        w["hist_len"] = rng.integers(0, hist - 1, rows).astype(np.uint32)
    if mask:
        words = (vocab + 31) // 32
        w["mask"] = rng.integers(0, 2**32, (rows, words), dtype=np.uint64).astype(np.uint32)
        w["mask"][1::3] = 0xFFFFFFFF
        w["mask"][:, 0] |= 1
    return w


def _masked(w):
    vocab = w["logits"].shape[1]
    return np.where(np.unpackbits(w["mask"].view(np.uint8), axis=1, bitorder="little")[:, :vocab] != 0, w["logits"], -np.inf)


@pytest.mark.parametrize("vocab", [2049, 16385, 65536])
@pytest.mark.parametrize("hist", [0, 200, 1100])
def test_masks_and_drafts(vocab, hist):
    rows = 70
    w = _batch(rows, vocab, 1, hist=hist)
    rng = np.random.Generator(np.random.PCG64([vocab, hist, 4]))
    draft = _masked(w).argmax(axis=1).astype(np.int32)
    draft[::3] = rng.integers(0, vocab, len(draft[::3]))
    u2 = workloads._uniforms(rng, rows)
    u2[::5] = np.float32(1.0 - 2.0**-24)
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab, max_hist=max(hist, 1))
    try:
        assert_parity(ctx, w, cap=64, hinted=True)
        g = gpu_rows(ctx, w, draft=draft, u2=u2, hinted=True)
        bad = [r for r, (t, tr) in enumerate(oracle_rows(w, draft=draft, u2=u2))
               if g["tokens"][r] != t or bool(g["accepted"][r]) != bool(tr["accepted"])]
        assert not bad, [(r, int(g["path"][r])) for r in bad[:8]]
    finally:
        ctx.close()


def test_histories_as_counts():
    rows, vocab, ids = 70, 40000, 150
    w = _batch(rows, vocab, 2, hist=0)
    w["params"]["repetition_penalty"], w["params"]["frequency_penalty"], w["params"]["presence_penalty"] = 1.1, 0.2, 0.3
    rng = np.random.Generator(np.random.PCG64([2, 5]))
    tokens = np.stack([rng.choice(vocab, ids, replace=False) for _ in range(rows)]).astype(np.int32)
    counts = rng.integers(0, 4, (rows, ids)).astype(np.uint32)
    length = rng.integers(0, ids + 1, rows).astype(np.uint32)
    plain = dict(w)
    plain["hist"] = np.zeros((rows, 3 * ids), np.int32)
    plain["hist_len"] = np.zeros(rows, np.uint32)
    for r in range(rows):
        t = np.repeat(tokens[r, :length[r]], counts[r, :length[r]])
        plain["hist"][r, :len(t)], plain["hist_len"][r] = t, len(t)
    w["hist"], w["hist_len"] = tokens, length
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab, max_hist=ids)
    try:
        g = gpu_rows(ctx, w, hist_counts=counts, hinted=True)
        ref = oracle_rows(plain)
        assert [int(t) for t in g["tokens"]] == [t for t, _ in ref]
        assert [int(n) for n in g["n_cand"]] == [tr["n_cand"] for _, tr in ref]
    finally:
        ctx.close()


def test_forced_and_close_tokens():
    """(and the chosen token appended to the row's history; twice, the second time with what the first has left)"""
    rows, vocab = 80, 33000
    w = _batch(rows, vocab, 3)
    rng = np.random.Generator(np.random.PCG64([3, 5]))
    masked = _masked(w)
    order = np.argsort(-masked, axis=1, kind="stable")
    force, close = np.full(rows, -1, np.int32), np.full(rows, -1, np.int32)
    force[::4] = rng.integers(0, vocab, len(force[::4]))
    close[1::3], close[2::6] = order[1::3, 1], order[2::6, 30]
    above = [int((masked[r] > masked[r, close[r]]).sum()) if close[r] >= 0 else 0xffffffff for r in range(rows)]
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab, max_hist=200)
    try:
        b = api.Batch(w["logits"], w["params"], w["u"], mask=w["mask"], hist=w["hist"], hist_len=w["hist_len"], force_token=force,
                      close_token=close, close_max_above=3, append_history=True, params_host=True)
        for _ in range(2):
            ref = oracle_rows(w)
            ctx.sample_batch(b.desc, params_host=b.params_host)
            g = b.results()
            taken = (close >= 0) & (np.array(above) < 3)
            want = np.where(force >= 0, force, np.where(taken, close, [t for t, _ in ref]))
            assert np.array_equal(g["tokens"], want), np.flatnonzero(g["tokens"] != want)[:8]
            assert np.array_equal(g["forced"] != api.FORCED_NONE, (force >= 0) | taken)
            for r in range(rows):
                w["hist"][r, w["hist_len"][r]] = want[r]
            w["hist_len"] += 1
            hist, length = b.history()
            assert np.array_equal(length, w["hist_len"]) and np.array_equal(hist, w["hist"])
    finally:
        ctx.close()


@pytest.mark.parametrize("vocab", [8191, 16387, 40960])
def test_rows_at_any_address(vocab):
    rows = 40
    w = _batch(rows, vocab, 4)
    ref = oracle_rows(w)
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab, max_hist=200)
    try:
        for pad, offset in ((0, 0), (1, 0), (64, 0), (0, 1), (2, 3), (4, 4)):
            flat = np.full(offset + rows * (vocab + pad) - pad, 1e30, np.float32)  # (the last row ends with the allocation)
            for r in range(rows):
                flat[offset + r * (vocab + pad):][:vocab] = w["logits"][r]
            buf = hip.DeviceArray.from_host(flat)
            b = api.Batch(w["logits"], w["params"], w["u"], mask=w["mask"], hist=w["hist"], hist_len=w["hist_len"], params_host=True)
            b.desc.logits, b.desc.logits_stride = buf.ptr + 4 * offset, vocab + pad
            ctx.sample_batch(b.desc, params_host=b.params_host)
            g = b.results()
            assert [int(t) for t in g["tokens"]] == [t for t, _ in ref], (pad, offset)
            assert [int(n) for n in g["n_cand"]] == [tr["n_cand"] for _, tr in ref], (pad, offset)
    finally:
        ctx.close()


@pytest.mark.parametrize("vocab", [700, 20000, 129280])
@pytest.mark.parametrize("rows", [9, 80])
def test_narrow_rows(vocab, rows):
    """Nuclei of a few up to some 300 tokens, finished from one to eight slices' candidate lists, or given back by them."""
    w = nucleus_batch(rows, vocab, vocab + 3, [2.0, 3.0, 4.0, 5.0, 6.0], [1.0, 0.8], [0.3, 0.6, 0.9], us=[0.0, 0.2, 0.7, 1.0 - 2.0**-24])
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)
    try:
        g = assert_parity(ctx, w, cap=300, hinted=True)
        assert (g["path"] == api.PATH_NUCLEUS).any()
    finally:
        ctx.close()


# (64 pieces of 8 192 logits at the most; beyond 262 144 a call without the host copy takes these kernels too, from 65 rows)
@pytest.mark.parametrize("vocab", [262144, 262145, 524288, 524289, 524292])
def test_long_rows(vocab):
    rows = 66
    w = nucleus_batch(rows, vocab, 9, [0.3, 1.0, 3.0, 6.0], [1.0, 0.7], [0.3, 0.9], us=[0.0, 0.3, 0.98])
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)
    try:
        for hinted in (True, False):
            assert_parity(ctx, w, cap=64, hinted=hinted)
    finally:
        ctx.close()


def test_random_batches():
    total = np.zeros(10, np.int64)
    for seed in range(9200, 9212):
        w, cap = random_large_batch(seed)
        b, v = w["logits"].shape
        ctx = api.SamplerContext(max_rows=b, max_vocab=v, max_hist=2048)
        try:
            g = assert_parity(ctx, w, cap=cap, hinted=True)
        finally:
            ctx.close()
        total += np.bincount(g["path"], minlength=10)
    assert total[api.PATH_SUMMED] > 100, total


def _checked(ctx, w, cap):
    ctx.failed_checks()  # (clears what an earlier batch left)
    g = assert_parity(ctx, w, cap=cap, hinted=True)
    bits = ctx.failed_checks()
    assert bits == CHECKED, "index checks failed: bit set 0x%x" % bits
    return g


@pytest.mark.parametrize("rows,vocab", [(6, 151552), (6, 196600), (40, 33000), (80, 2049), (140, 65537), (66, 262144)])
def test_no_index_check_fails(rows, vocab):
    w = _batch(rows, vocab, 6, mask=rows != 140)
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab, max_hist=200, lib_path=api.CHECKED_LIB_PATH)
    try:
        _checked(ctx, w, 64)
    finally:
        ctx.close()


def test_no_index_check_fails_on_flat_and_peaked_rows():
    ctx = api.SamplerContext(max_rows=256, max_vocab=151552, lib_path=api.CHECKED_LIB_PATH)
    try:
        g = _checked(ctx, workloads.config4(), 64)
        assert (g["path"] == api.PATH_SUMMED).any()
    finally:
        ctx.close()


def test_rash_plans():
    """Shares left unsorted that should not be: the tail gives such rows up, and finishes others on records that held."""
    ctx = api.SamplerContext(max_rows=256, max_vocab=262144, lib_path=api.RASH_LIB_PATH)
    us = [0.0, 1e-4, 0.1, 0.25, 0.5, 0.6, 0.7, 0.8, 0.9, 0.95, 0.99, 0.9999, 1.0 - 2.0**-24]
    try:
        g = _checked(ctx, workloads.config4(), 256)
        assert (g["path"] == api.PATH_GENERAL).any() and (g["path"] == api.PATH_SUMMED).any()
        _checked(ctx, nucleus_batch(136, 129280, 12, sigmas=[0.1, 1.0], temps=[1.0], top_ps=[0.9, 0.97], us=us), 64)
        _checked(ctx, nucleus_batch(40, 262144, 13, sigmas=[0.05, 0.3], temps=[1.0], top_ps=[0.9, 0.999], us=us), 64)
        g = _checked(ctx, nucleus_batch(160, 129280, 11, sigmas=[0.05, 0.1, 0.3, 1.0, 2.0, 3.0, 0.2], temps=[0.5, 1.0, 1.5],
                                        top_ps=[0.5, 0.9, 0.99, 0.999, 0.8]), 128)
        assert (g["path"] == api.PATH_GENERAL).any()
    finally:
        ctx.close()


def test_rash_plans_of_random_batches():
    total = np.zeros(10, np.int64)
    for seed in range(9300, 9308):
        w, cap = random_large_batch(seed)
        b, v = w["logits"].shape
        ctx = api.SamplerContext(max_rows=b, max_vocab=v, max_hist=2048, lib_path=api.RASH_LIB_PATH)
        try:
            g = _checked(ctx, w, cap)
        finally:
            ctx.close()
        total += np.bincount(g["path"], minlength=10)
    assert total[api.PATH_GENERAL] > 30, total
