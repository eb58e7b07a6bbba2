"""GPU parity of the rounds of std::ranges::nth_element that several workgroups make of a long row (nth_steps.h): rows that are
their own list and rows with gaps, where the rounds stop (a cut in front of top_k, a top_k beyond the candidates), pivots that
are penalised or change places, in launches of their own and beside other rows."""
import numpy as np
import pytest

from mako_amd import api
from parity import assert_parity, gpu_rows, oracle_rows

pytestmark = pytest.mark.gpu


def _batch(vocab, gaps, seed, ties, hist=0):
    rng = np.random.Generator(np.random.PCG64([seed, vocab, hist]))
    top_ks = [1, 2, 40, 300, 16380, vocab // 2, vocab - 1, vocab, 2 * vocab]
    rows = len(top_ks)
    x = (rng.standard_normal((rows, vocab)) * 2.0).astype(np.float32)
    if ties:
        x = np.round(x * 4.0) / np.float32(4.0)
    x[2, vocab // 2] = x[2, 1] = x[2, -1] = 9.0  # (a row whose first pivot is its best entry)
    p = api.make_params(rows, 0.8, 0, 1.0)
    p["top_k"] = top_ks
    p["top_p"][3] = np.float32(0.97)  # (survivors that are sorted)
    w = dict(name="V=%d %s" % (vocab, gaps), logits=x, params=p, u=rng.random(rows).astype(np.float32))
    if gaps == "mask":
        m = rng.integers(0, 2**32, (rows, (vocab + 31) // 32), dtype=np.uint64).astype(np.uint32)
        m[1] = 0
        m[1, 5] = 0x10  # (a row with one candidate)
        m[5] = 0xFFFFFFFF
        w["mask"] = m
    elif gaps == "min_p":
        p["min_p"] = np.float32(1e-3)
    elif gaps == "underflow":  # whole stretches with a weight of zero, the row's first entries among them
        x[:, : vocab // 3] = -500.0
        x[::2, -100:] = -np.inf
    elif gaps == "one":  # a single entry missing: the last, the middle or the first
        for r in range(rows):
            x[r, (vocab - 1, vocab // 2, 0)[r % 3]] = -np.inf
    if hist:
        for name, v in (("repetition_penalty", 1.3), ("frequency_penalty", 0.2), ("presence_penalty", 0.3)):
            p[name] = np.float32(v)
        h = rng.integers(0, vocab, (rows, hist)).astype(np.int32)
        h[:, :6] = [0, 1, vocab // 2, vocab - 1, 1, vocab // 2]
        w["hist"], w["hist_len"] = h, np.full(rows, hist, np.uint32)
        w["hist_len"][0] = 3
    return w


# (there are no steps up to 32 768 logits: rows of 16 381 and 20 002 take the same rounds in the last launch alone, more than its
# registers hold and no more)
@pytest.mark.parametrize("gaps", ["none", "mask", "min_p", "underflow", "one"])
@pytest.mark.parametrize("vocab", [16381, 20002, 65537, 131072, 151553])
def test_steps(vocab, gaps):
    ctx = api.SamplerContext(max_rows=16, max_vocab=vocab, max_hist=64)
    try:
        for ties in (False, True):
            w = _batch(vocab, gaps, 3, ties, hist=20 if ties else 0)
            for hinted in (True, False):
                assert_parity(ctx, w, cap=64, hinted=hinted)
            # beside a nucleus, a row in token order and a top-k row
            w["params"]["top_k"][4:7] = (0, 0, 30)
            w["params"]["top_p"][4:7] = (0.9, 1.0, 0.9)
            for hinted in (True, False):
                assert_parity(ctx, w, cap=64, hinted=hinted)
    finally:
        ctx.close()


@pytest.mark.parametrize("vocab", [20002, 151552])
def test_steps_forced_and_verified(vocab):
    w = _batch(vocab, "mask", 4, True)
    rows = len(w["u"])
    rng = np.random.Generator(np.random.PCG64(vocab))
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)
    try:
        force = np.full(rows, -1, np.int32)
        force[[2, 6]] = (7, 11)
        for hinted in (True, False):
            g = api.sample(ctx, w["logits"], w["params"], w["u"], mask=w["mask"], force_token=force, params_host=hinted)
            ref = oracle_rows(w)
            for r in range(rows):
                assert g["tokens"][r] == (force[r] if force[r] >= 0 else ref[r][0]), (r, hinted)
        draft = rng.integers(0, vocab, rows).astype(np.int32)
        draft[::2] = np.where(w["logits"].max(1, keepdims=True) == w["logits"], np.arange(vocab), -1).max(1)[::2]
        u2 = rng.random(rows).astype(np.float32)
        for hinted in (True, False):
            g = gpu_rows(ctx, w, draft=draft, u2=u2, hinted=hinted)
            for r, (t, tr) in enumerate(oracle_rows(w, draft=draft, u2=u2)):
                assert (g["tokens"][r], bool(g["accepted"][r])) == (t, bool(tr["accepted"])), (r, hinted)
    finally:
        ctx.close()


# (launches of their own with two steps at most, of rows with and without gaps, whose first pivots are penalised or not; and the
# longest rows without steps and with two)
@pytest.mark.parametrize("gaps", ["none", "mask", "min_p", "underflow", "one"])
@pytest.mark.parametrize("vocab", [32768, 32769, 40000, 50001, 65536])
def test_two_steps(vocab, gaps):
    test_steps(vocab, gaps)
    w = _batch(vocab, gaps, 6, False, hist=30)  # (the least top_k of a batch says how many launches it takes)
    ctx = api.SamplerContext(max_rows=len(w["u"]), max_vocab=vocab, max_hist=64)
    try:
        for first in (4, 5, 7):
            part = {k: v if k == "name" else v[first:] for k, v in w.items()}
            assert_parity(ctx, part, cap=64, hinted=True)
    finally:
        ctx.close()


@pytest.mark.parametrize("vocab", [32769, 40000, 65536])
def test_two_steps_forced_and_verified(vocab):
    test_steps_forced_and_verified(vocab)


# (the bin that holds the k-th heaviest: a few entries more than k, thousands, more than one sort in LDS holds)
@pytest.mark.parametrize("vocab", [2048, 2049, 9001, 16381, 40000, 131072, 151553])
@pytest.mark.parametrize("sigma", [3.0, 0.5, 0.02])
def test_wide_top_k_before_a_top_p(vocab, sigma):
    rng = np.random.Generator(np.random.PCG64([vocab, int(sigma * 100)]))
    top_ks = [k for k in (129, 200, 500, 1000, 4096, 6143, 6144, 6145, 9000) if k < vocab] + [vocab - 1, vocab]
    rows = len(top_ks)
    x = (rng.standard_normal((rows, vocab)) * sigma).astype(np.float32)
    x[1::3] = np.round(x[1::3] * 16.0) / np.float32(16.0)
    p = api.make_params(rows, 1.0, 0, 0.95)
    p["top_k"] = top_ks
    p["top_p"][::2] = np.float32(0.9999)
    p["min_p"][3] = np.float32(0.5)
    w = dict(name="wide V=%d" % vocab, logits=x, params=p, u=rng.random(rows).astype(np.float32))
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)
    try:
        for masked in (False, True):
            if masked:
                w["mask"] = rng.integers(0, 2**32, (rows, (vocab + 31) // 32), dtype=np.uint64).astype(np.uint32)
            for hinted in (True, False):
                assert_parity(ctx, w, cap=300, hinted=hinted)
        p["top_k"][0], p["top_p"][0] = 0, 0.9  # (beside a nucleus)
        for hinted in (True, False):
            assert_parity(ctx, w, cap=300, hinted=hinted)
    finally:
        ctx.close()


# (beside other rows a row's workgroups make all steps in one launch and wait for each other in between; in the checked build
# those of every other row don't, and leave the rest to the last launch)
@pytest.mark.parametrize("checked", [False, True])
@pytest.mark.parametrize("vocab, copies", [(32769, 1), (32769, 8), (40000, 34), (151553, 1)])
def test_steps_in_one_launch(vocab, copies, checked):
    ctx = api.SamplerContext(max_rows=9 * copies, max_vocab=vocab, lib_path=api.CHECKED_LIB_PATH if checked else None)
    try:
        for gaps in ("none", "mask"):
            w = _batch(vocab, gaps, 5, False)
            if copies > 1:  # (the same rows again; many have one workgroup each)
                w = {k: v if k == "name" else np.concatenate([v] * copies) for k, v in w.items()}
            one = oracle_rows({k: v if k == "name" else v[:9] for k, v in w.items()}, cap=64)
            if checked:
                ctx.failed_checks()
            for _ in range(3):
                g = gpu_rows(ctx, w, cap=64, hinted=False)
                for r in range(9 * copies):
                    t, tr = one[r % 9]
                    n = min(64, tr["n_cand"])
                    assert (g["tokens"][r], g["n_cand"][r]) == (t, tr["n_cand"]), (r, gaps)
                    assert np.array_equal(g["cand_idx"][r, :n], tr["cand_idx"][:n]), (r, gaps)
                    assert np.float32(g["total"][r]).view(np.uint32) == np.float32(tr["total"]).view(np.uint32), (r, gaps)
            if checked:
                assert ctx.failed_checks() == 1 << 31
    finally:
        ctx.close()
