"""GPU parity of rows whose nucleus ends in a light tail behind a bin that holds nearly all of the row's mass, with top_p within a few
units of fp32 of one: the plan's estimate of what lies below a bin may not lose that tail."""
import numpy as np
import pytest

from mako_amd import api, workloads
from parity import assert_parity

pytestmark = pytest.mark.gpu

UNITS = 256  # of the plan's bins in a factor of two of the weight
FINE, GROUP = 512, 16  # bins of one unit, and units of a bin behind them


def _logit(b):
    """The middle of bin b, b >= FINE, of a row whose maximum is the middle of its unit."""
    unit = -FINE // GROUP - (b - FINE)  # group number; (the maximum's unit is 0)
    return (unit * GROUP + GROUP // 2) / UNITS * np.log(2.0)


@pytest.mark.parametrize("rows", [4, 40])
def test_tails_behind_a_heavy_bin(rows):
    rng = np.random.Generator(np.random.PCG64([rows, 5]))
    vocab = 200000
    logits = np.empty((rows, vocab), np.float32)
    p = workloads.make_params(rows, 1.0, 0, 0.9)
    for r in range(rows):
        one_less = [2.0**-23, 2.0**-22, 2.0**-21, 2.0**-20][r % 4]
        heavy = FINE + 2 * int(rng.integers(1, 190))
        n = int(rng.integers(120000, 190000))
        mass = 1.0 + n * np.exp(_logit(heavy))
        want, tail = one_less * mass * 1.5, []
        for _ in range(400):  # the tail: weights of up to what is left of half as much again as may be left out
            b = int(rng.integers(heavy + 60, min(heavy + 129, 1020)))
            if np.exp(_logit(b)) < want:
                want -= np.exp(_logit(b))
                tail.append(_logit(b))
        row = np.full(vocab, -1e4)
        row[:n] = _logit(heavy)
        row[n], row[n + 1] = 0.5 / UNITS * np.log(2.0), _logit(heavy + 1)
        row[n + 2:n + 2 + len(tail)] = tail
        logits[r] = rng.permutation(row)
        p["top_p"][r] = np.float32(1.0) - np.float32(one_less)
    w = dict(name="tails", logits=logits, params=p, u=rng.random(rows).astype(np.float32))
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)
    try:
        for hinted in (True, False):
            g = assert_parity(ctx, w, cap=64, hinted=hinted)
            print(np.bincount(g["path"], minlength=9).tolist(), flush=True)
    finally:
        ctx.close()
