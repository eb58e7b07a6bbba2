"""Verification (src/gen/sampler.cpp:86-107) of rows that end in a short sorted list: one wave accepts or redraws."""
import numpy as np
import pytest

from mako_amd import api
from parity import gpu_rows, oracle_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [37, 4099, 129280])
@pytest.mark.parametrize("top_k", [0, 1, 2, 63, 64, 65, 128])
def test_drafts_everywhere_in_a_short_list(gpu_ctx, vocab, top_k):
    """Drafts at the list's first and last place and in between, outside it, and as the only candidate; accepted,
    and rejected with the redraw's uniform at its ends (top_k 0: a nucleus of a few tokens)."""
    rows = 24
    rng = np.random.default_rng([vocab, top_k])
    logits = (rng.standard_normal((rows, vocab)) * 3.0).astype(np.float32)
    p = api.make_params(rows, 0.8, top_k, 0.95)
    if top_k == 0:
        p["temperature"], p["top_p"] = 0.2, 0.9
    u = np.where(np.arange(rows) % 3 == 0, 0.0, rng.random(rows)).astype(np.float32)
    u[1::6] = np.float32(1.0 - 2.0**-24)
    u2 = np.where(np.arange(rows) % 4 == 0, 0.0, rng.random(rows)).astype(np.float32)
    u2[1::4] = np.float32(1.0 - 2.0**-24)
    w = dict(name="short verify", logits=logits, params=p, u=u)
    drafts = np.empty(rows, np.int32)
    for r, (_, tr) in enumerate(oracle_rows(w, cap=128)):
        ids = tr["cand_idx"][:min(128, tr["n_cand"])]
        drafts[r] = [ids[0], ids[-1], ids[len(ids) // 2], rng.integers(0, vocab)][r % 4]
    g = gpu_rows(gpu_ctx, w, draft=drafts, u2=u2, hinted=top_k != 0)
    for r, (t, tr) in enumerate(oracle_rows(w, draft=drafts, u2=u2)):
        assert g["tokens"][r] == t and bool(g["accepted"][r]) == bool(tr["accepted"]), (r, int(drafts[r]), g["tokens"][r], t)
    if top_k:
        assert (g["path"] == api.PATH_TOPK).all()
