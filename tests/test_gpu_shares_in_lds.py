"""GPU parity of flat rows with the host copy of the parameters, whose workers sort in workgroups of 512 threads: shares of up to 5 120
entries (a copy of the sorted weights beside the sort), up to 6 144 (the copy over the entries), and beyond (in runs); with none, few
and many equal weights, in batches whose workers all sort and in ones that leave shares unsorted."""
import numpy as np
import pytest

from mako_amd import api
from parity import assert_parity, nucleus_batch

pytestmark = pytest.mark.gpu


# (32 workers of 5 120 entries hold 163 840, of 6 144 196 608)
@pytest.mark.parametrize("rows", [6, 40])
@pytest.mark.parametrize("grid", [0.0, 2.0**-9, 2.0**-5])
@pytest.mark.parametrize("vocab", [520, 4200, 17000, 129280, 151552, 163800, 167000, 181000, 196600, 204000, 230000])
def test_flat_rows(vocab, grid, rows):
    w = nucleus_batch(rows, vocab, vocab + rows, [0.05, 0.6, 2.5], [1.0, 0.7], [0.9995, 0.97], us=[0.3, 0.98, 0.0])
    if grid:
        w["logits"] = (np.round(w["logits"] / grid) * grid).astype(np.float32)
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)
    try:
        assert_parity(ctx, w, cap=min(vocab, 20000) if rows == 6 else 64, hinted=True)
    finally:
        ctx.close()


@pytest.mark.parametrize("above", [0.5, 1.0, 2.0, 4.0, 8.0])
@pytest.mark.parametrize("vocab", [182000, 188000, 194000, 230000])
def test_crowded_shares(vocab, above):
    """One token far above the others: the share it is in has a wide range of weights, nearly all of them at its lower end, in buckets
    too crowded for one sort, for a run's, or for neither."""
    for rows in (6, 36):
        w = nucleus_batch(rows, vocab, vocab + int(above * 2), [0.1, 0.05, 0.3], [1.0], [0.9999], us=[0.3, 0.98, 0.0])
        at = np.arange(rows) * 4099 % vocab
        w["logits"][np.arange(rows), at] = w["logits"].max(axis=1) + np.float32(above)
        ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)
        try:
            assert_parity(ctx, w, cap=12000, hinted=True)
        finally:
            ctx.close()
