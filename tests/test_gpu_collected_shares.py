"""GPU parity of large batches whose flat rows leave from a few to some two dozen shares unsorted: the workgroups that take them
have eight waves with a share each or, from 81 rows, two (with the host copy of the parameters), or sixteen (without it)."""
import pytest

from mako_amd import api
from parity import assert_parity, nucleus_batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [41000, 74000, 107000, 129280, 196000, 262144])
@pytest.mark.parametrize("rows", [66, 80, 81])
def test_one_to_four_workgroups_a_row(vocab, rows):
    w = nucleus_batch(rows, vocab, vocab + 5, [0.05, 0.1, 0.4], [1.0], [0.9, 0.9995], us=[0.0, 0.3, 0.98, 1.0 - 2.0**-24, 0.6])
    w["params"]["top_k"][5::11] = 40
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)
    try:
        for hinted in (True, False):
            g = assert_parity(ctx, w, cap=64, hinted=hinted)
            assert (g["path"] == api.PATH_SUMMED).any()
    finally:
        ctx.close()
