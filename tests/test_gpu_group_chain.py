"""The exact fp32 total and walk of long lists (mako_amd/csrc/group_chain.h): what a group of 256 weights adds as one
number, the replay of groups in which the binade changes, exact ties, and the staged head of the list."""
import numpy as np
import pytest

from mako_amd import api
from parity import assert_parity

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
