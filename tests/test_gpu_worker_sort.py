"""GPU parity of the workers' sorts of a wide nucleus: shares around what one sort in LDS holds, shares cut into runs, weights that
crowd few buckets, and rows whose list is shared out to one worker, a few or all of them."""
import numpy as np
import pytest

from mako_amd import api
from parity import assert_parity, nucleus_batch

pytestmark = pytest.mark.gpu


# (32 workers of 6 144 entries in LDS hold 196 608, of 5 632 180 224; a worker is given 512 entries at least, 4 096 on a large batch)
@pytest.mark.parametrize("vocab", [520, 1030, 4200, 17000, 176000, 181000, 196000, 199000, 230000, 260000])
@pytest.mark.parametrize("grid", [0.0, 2.0**-9, 2.0**-5])
def test_flat_rows(vocab, grid):
    rows = 6
    w = nucleus_batch(rows, vocab, vocab, [0.05, 0.4, 1.5], [1.0], [0.97, 0.9995], us=[0.0, 0.3, 0.98])
    if grid:
        w["logits"] = (np.round(w["logits"] / grid) * grid).astype(np.float32)
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)
    try:
        for hinted in (True, False):
            assert_parity(ctx, w, cap=3000, hinted=hinted)
    finally:
        ctx.close()


@pytest.mark.parametrize("vocab", [4200, 9000, 30000])
def test_large_batches_of_short_lists(vocab):
    rows = 96
    w = nucleus_batch(rows, vocab, vocab + 1, [0.05, 0.4, 1.5, 4.0], [1.0, 0.6], [0.5, 0.9, 0.999])
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)
    try:
        for hinted in (True, False):
            assert_parity(ctx, w, cap=64, hinted=hinted)
    finally:
        ctx.close()


@pytest.mark.parametrize("vocab", [176000, 181000, 230000])
@pytest.mark.parametrize("grid", [0.0, 2.0**-6])
def test_large_batches_of_flat_rows(vocab, grid):
    rows = 66
    w = nucleus_batch(rows, vocab, vocab + 2, [0.05, 0.6, 2.5], [1.0], [0.97, 0.9995], us=[0.0, 0.3, 0.98])
    if grid:
        w["logits"] = (np.round(w["logits"] / grid) * grid).astype(np.float32)
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)
    try:
        assert_parity(ctx, w, cap=64, hinted=True)
    finally:
        ctx.close()


def test_narrow_rows_of_a_large_batch():
    """Nuclei of a few up to some 300 tokens, finished from one to eight slices' candidate lists."""
    for vocab in (700, 20000, 129280):
        rows = 80
        w = nucleus_batch(rows, vocab, vocab + 3, [2.0, 3.0, 4.0, 5.0, 6.0], [1.0, 0.8], [0.3, 0.6, 0.9], us=[0.0, 0.2, 0.7, 1.0 - 2.0**-24])
        ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)
        try:
            g = assert_parity(ctx, w, cap=300)
            assert (g["path"] == api.PATH_NUCLEUS).any()
        finally:
            ctx.close()
