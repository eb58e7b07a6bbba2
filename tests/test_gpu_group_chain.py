"""The exact fp32 total and walk of long lists (mako_amd/csrc/group_chain.h): what a group of 256 weights adds as one
number, the replay of groups in which the binade changes, exact ties, and the staged head of the list."""
import numpy as np
import pytest

from mako_amd import api
from parity import assert_parity, gpu_rows, oracle_rows

pytestmark = pytest.mark.gpu


def _logits(kind, rows, vocab, rng):
    if kind == "equal":  # every weight 1: each addition is a tie or exact, the sum changes binade at every power of two
        return np.zeros((rows, vocab), np.float32)
    x = rng.standard_normal((rows, vocab))
    if kind == "grid":  # a handful of distinct weights
        return (np.round(x * 2) / 2).astype(np.float32)
    if kind == "peaked":  # one weight near 1, the others far below: the sum's first binades pass in one group
        x *= 0.05
        x[:, vocab // 3] += 12.0
        return x.astype(np.float32)
    return (x * 1.5).astype(np.float32)


# one entry short of, at and behind: the lists that go entry by entry, the staged head, a whole number of groups, the
# blocks of 64 groups
@pytest.mark.parametrize("vocab", [1020, 1024, 1025, 3068, 3072, 3073, 3328, 16384, 16385, 65540])
@pytest.mark.parametrize("kind", ["equal", "grid", "peaked", "normal"])
@pytest.mark.parametrize("top_p", [1.0, 0.999])
def test_totals_and_walks(gpu_ctx, vocab, kind, top_p):
    us = np.array([0.0, 2.0**-24, 0.1, 0.3, 0.5, 0.77, 0.9, 0.99, 0.999, 1.0 - 2.0**-24], np.float32)
    rng = np.random.default_rng([vocab, len(kind)])
    rows = len(us)
    w = dict(name="%s %d" % (kind, vocab), logits=_logits(kind, rows, vocab, rng), u=us,
             params=api.make_params(rows, np.linspace(0.6, 1.4, rows), 0, top_p))
    assert_parity(gpu_ctx, w, cap=64, hinted=True)


@pytest.mark.parametrize("vocab", [9000, 129280])
@pytest.mark.parametrize("hinted", [False, True])
def test_walks_in_the_lowest_binade(gpu_ctx, vocab, hinted):
    """A weight in [2^-126, 2^-125) far in front of the only other one, 1.0, and a walk that starts one last place below
    it, at it, above it, and at the ends of the binade: sums with such a weight lie in the next binade, whose last place is
    twice as large."""
    at = 5000
    r = [float.fromhex(x + "p-126") for x in ("0x1.01b1b8", "0x1.01b1ba", "0x1.01b1bc", "0x1.fffffe")]
    r += [2.0**-126, 2.0**-127, 2.0**-149, 0.0, 0.5]
    u = np.array(r, np.float32)
    logits = np.full((len(r), vocab), -np.inf, np.float32)
    logits[:, at] = np.float32(-87.3299484)
    logits[:, -1] = 0.0
    w = dict(name="lowest binade", logits=logits, u=u, params=api.make_params(len(r), 1.0, 0, 1.0))
    ref = oracle_rows(w, cap=4)
    assert ref[0][1]["cand_q"][0] == np.float32(float.fromhex("0x1.01b1bap-126"))
    assert [t for t, _ in ref] == [at, vocab - 1, vocab - 1, vocab - 1, at, at, at, at, vocab - 1]
    g = assert_parity(gpu_ctx, w, cap=0, hinted=hinted)
    assert (g["n_cand"] == 2).all()


@pytest.mark.parametrize("rows", [24, 64])
@pytest.mark.parametrize("hinted", [False, True])
def test_running_sum_ahead_of_its_estimates(rows, hinted):
    """Two weights near 1 and a tail of weights of about 2^-24, in a sum just below 2: each is rounded up or down to a whole
    last place, so that the running sum passes 2 dozens of groups before or behind the fp64 sums, which in some of the larger
    batch's rows pass it a few groups away from where the plan's estimates do.  The increments of those groups are for neither
    the binade that is expected in the end nor, maybe, for the one that the running sum is in."""
    vocab = 65540
    rng = np.random.default_rng([rows, 11])
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)
    logits = np.empty((rows, vocab), np.float32)
    for r in range(rows):
        c = [0.55, 0.8, 1.1, 1.4, 1.6, 1.9][r % 6] * (1.0 + 0.02 * rng.random())
        mass = vocab * c * 2.0**-24
        heads = rng.uniform(0.01, 0.02, r % 5)
        second = 1.0 - heads.sum() - mass * rng.uniform(0.1, 0.9)
        logits[r] = np.log(c * 2.0**-24) + 1e-3 * rng.standard_normal(vocab)
        at = rng.permutation(vocab)[:2 + len(heads)]
        logits[r, at] = np.log(np.concatenate([[1.0, second], heads]))
    u = rng.random(rows).astype(np.float32)
    u[::2] = np.float32(1.0) - rng.uniform(0.0, 2e-3, len(u[::2])).astype(np.float32)
    w = dict(name="ahead of its estimates", logits=logits, u=u, params=api.make_params(rows, 1.0, 0, 1.0))
    try:
        for top_p in (1.0, 1.0 - 2.0**-20):
            w["params"]["top_p"] = np.float32(top_p)
            assert_parity(ctx, w, cap=0, hinted=hinted)
    finally:
        ctx.close()


@pytest.mark.parametrize("masked", [3072, 3073, 20000, 65536, 129278])
def test_walks_from_zero_behind_a_masked_stretch(gpu_ctx, masked):
    """u = 0 and the first tokens masked: the walk passes every group in front of the first candidate at r = 0."""
    rng = np.random.default_rng(masked)
    rows, vocab = 6, 129280
    logits = (rng.standard_normal((rows, vocab)) * 2.0).astype(np.float32)
    logits[:, :masked] = -np.inf
    logits[3, 5] = 3.0  # (one row with a candidate in front of the stretch, drawn behind it)
    u = np.array([0.0, 0.0, 2.0**-24, 0.9, 0.5, 2.0**-149], np.float32)
    w = dict(name="from zero", logits=logits, u=u, params=api.make_params(rows, 1.0, 0, 1.0))
    draft = np.array([masked, vocab - 1, masked + 1, 5, 0, masked], np.int32)
    assert_parity(gpu_ctx, w, cap=0, hinted=True)
    assert_parity(gpu_ctx, w, cap=0)
    for u2 in (np.zeros(rows, np.float32), u):
        g = gpu_rows(gpu_ctx, w, draft=draft, u2=u2, hinted=True)
        for r, (t, tr) in enumerate(oracle_rows(w, draft=draft, u2=u2)):
            assert g["tokens"][r] == t and bool(g["accepted"][r]) == bool(tr["accepted"]), (r, g["tokens"][r], t)


@pytest.mark.parametrize("first", [3070, 3071, 3072, 3200, 3385, 65536, 129000])
@pytest.mark.parametrize("hinted", [False, True])
def test_redraws_from_zero_behind_the_staged_head(gpu_ctx, first, hinted):
    """A rejected draft that is the row's first candidate, behind the part of the list that is kept in LDS, and a redraw from
    u2 = 0: the walk passes the head at r = 0 and must not find the draft in its group's entries, which were fetched for
    the sum."""
    rng = np.random.default_rng(first)
    rows, vocab = 8, 129280
    logits = np.full((rows, vocab), -np.inf, np.float32)
    logits[:, first] = rng.uniform(-1.0, 1.0, rows)
    for r in range(rows):
        others = rng.integers(first + 1, vocab, 2 + 40 * r)
        logits[r, others] = rng.uniform(-2.0, 2.0, len(others))
    u = np.linspace(0.6, 0.99, rows).astype(np.float32)
    w = dict(name="redraw from zero", logits=logits, u=u, params=api.make_params(rows, 1.0, 0, 1.0))
    draft = np.full(rows, first, np.int32)
    for u2 in (np.zeros(rows, np.float32), np.full(rows, 2.0**-149, np.float32), np.full(rows, 2.0**-24, np.float32)):
        g = gpu_rows(gpu_ctx, w, draft=draft, u2=u2, hinted=hinted)
        for r, (t, tr) in enumerate(oracle_rows(w, draft=draft, u2=u2)):
            assert g["tokens"][r] == t and bool(g["accepted"][r]) == bool(tr["accepted"]), (r, g["tokens"][r], t)
