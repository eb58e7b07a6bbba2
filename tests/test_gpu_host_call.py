"""mako_sampler_sample_host() against the call on device pointers: inputs of every size on their way through the staging
memory (copies of 1 MiB, 16 MiB of pinned memory that is used again), rows apart from each other, histories as pairs; and on a
system that has no pinned memory to give."""
import ctypes

import numpy as np
import pytest

from mako_amd import api, workloads
from parity import gpu_rows

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,vocab,apart", [(1, 1, 0), (1, 3, 5), (3, 4099, 0), (2, 131072, 0), (5, 65536, 64), (1, 262145, 0), (33, 140001, 3)])
@pytest.mark.parametrize("verify", [False, True])
@pytest.mark.parametrize("lib", [api.LIB_PATH, api.RASH_LIB_PATH], ids=["pinned", "no pinned memory"])
def test_same_as_the_device_call(rows, vocab, apart, verify, lib):
    rng = np.random.Generator(np.random.PCG64([rows, vocab]))
    whole = (rng.standard_normal((rows, vocab + apart)) * 3.0).astype(np.float32)
    p = api.make_params(rows, 0.8, 40, 0.95)
    p["repetition_penalty"], p["frequency_penalty"], p["presence_penalty"] = 1.1, 0.2, 0.3
    p["temperature"][::5] = 0.0
    n = min(vocab, 300)
    hist = np.stack([rng.permutation(vocab)[:n] for _ in range(rows)]).astype(np.int32)
    counts = rng.integers(1, 4, (rows, n)).astype(np.uint32)
    length = rng.integers(0, n + 1, rows).astype(np.uint32)
    words = (vocab + 31) // 32
    mask = rng.integers(0, 1 << 32, (rows, words + 1), dtype=np.uint64).astype(np.uint32)
    mask[:, 0] |= 1
    u, u2 = workloads._uniforms(rng, rows), workloads._uniforms(rng, rows)
    draft = rng.integers(0, vocab, rows).astype(np.int32)
    tokens, accepted = np.full(rows, -1, np.int32), np.zeros(rows, np.uint8)
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab, max_hist=512, lib_path=lib)

    def at(a):
        return ctypes.c_void_p(a.ctypes.data)

    try:
        for _ in range(2):
            rc = ctx.lib.mako_sampler_sample_host(
                ctypes.c_void_p(ctx.ptr), at(whole), vocab + apart, rows, vocab, at(p), at(u), at(mask), words + 1, at(hist), at(counts), n,
                at(length), at(draft) if verify else None, at(u2) if verify else None, at(accepted) if verify else None, at(tokens))
            assert rc == api.MAKO_OK, ctx.last_error()
            w = dict(logits=np.ascontiguousarray(whole[:, :vocab]), params=p, u=u, mask=np.ascontiguousarray(mask[:, :words]), hist=hist,
                     hist_len=length)
            g = gpu_rows(ctx, w, hist_counts=counts, draft=draft if verify else None, u2=u2 if verify else None)
            assert np.array_equal(tokens, g["tokens"])
            if verify:
                assert np.array_equal(accepted, g["accepted"])
            whole[:] = np.roll(whole, 1, axis=1)
    finally:
        ctx.close()


# (top-k and greedy rows whose inputs would be one copy are read where they were put together: also where the candidates don't
# settle a row, whose logits are then read again, and on either side of a MiB)
@pytest.mark.parametrize("rows,vocab", [(1, 8), (1, 129280), (4, 32000), (1, 261800), (1, 262100), (1, 262200)])
def test_inputs_left_in_place(rows, vocab):
    rng = np.random.Generator(np.random.PCG64([rows, vocab]))
    tokens = np.full(rows, -1, np.int32)
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab)

    def at(a):
        return ctypes.c_void_p(a.ctypes.data)

    try:
        for top_k, top_p, levels in ((40, 0.95, 0), (40, 0.95, 1), (128, 0.999, 3), (0, 0.9, 0)):
            x = (rng.standard_normal((rows, vocab)) * 3.0).astype(np.float32)
            if levels:
                x = np.floor(x.clip(0, levels - 0.5))
            p = api.make_params(rows, 0.8, top_k, top_p)
            p["temperature"][1:2] = 0.0
            u = rng.random(rows).astype(np.float32)
            rc = ctx.lib.mako_sampler_sample_host(ctypes.c_void_p(ctx.ptr), at(x), vocab, rows, vocab, at(p), at(u), None, 0, None, None, 0, None, None,
                                                  None, None, at(tokens))
            assert rc == api.MAKO_OK, ctx.last_error()
            assert np.array_equal(tokens, gpu_rows(ctx, dict(logits=x, params=p, u=u))["tokens"]), (top_k, levels)
    finally:
        ctx.close()


# (on either side of the 16 KiB up to which a call is copied all the same)
@pytest.mark.parametrize("rows,vocab", [(1, 3964), (1, 3968), (1, 3969), (1, 3972), (16, 200), (16, 260)])
def test_small_calls(rows, vocab):
    test_inputs_left_in_place(rows, vocab)


# (rows whose histories are long enough to be read in trips go through a copy, and greedy rows and rows without penalties, which have
# no use for theirs, don't: around the 8 192 entries that a slice's threads hold in registers, with rows that are read again)
@pytest.mark.parametrize("entries", [1, 8191, 8192, 8193, 20000])
@pytest.mark.parametrize("vocab", [9000, 40001])
def test_long_histories(vocab, entries):
    rows = 3
    rng = np.random.Generator(np.random.PCG64([vocab, entries]))
    tokens = np.full(rows, -1, np.int32)
    ctx = api.SamplerContext(max_rows=rows, max_vocab=vocab, max_hist=20000)

    def at(a):
        return ctypes.c_void_p(a.ctypes.data)

    try:
        for levels in (0, 2):
            x = (rng.standard_normal((rows, vocab)) * 3.0).astype(np.float32)
            if levels:
                x = np.floor(x.clip(0, levels - 0.5))
            p = api.make_params(rows, 0.8, 40, 0.95)
            hist = rng.integers(0, vocab, (rows, entries)).astype(np.int32)
            counts = rng.integers(1, 4, (rows, entries)).astype(np.uint32)
            length = np.array([entries, entries // 2, entries], np.uint32)
            u = rng.random(rows).astype(np.float32)
            for penalised in ((), (0,), (0, 1, 2)):
                p["repetition_penalty"][list(penalised)], p["frequency_penalty"][list(penalised)] = 1.3, 0.2
                p["temperature"][2] = 0.0 if len(penalised) == 1 else 0.8
                rc = ctx.lib.mako_sampler_sample_host(ctypes.c_void_p(ctx.ptr), at(x), vocab, rows, vocab, at(p), at(u), None, 0, at(hist),
                                                      at(counts), entries, at(length), None, None, None, at(tokens))
                assert rc == api.MAKO_OK, ctx.last_error()
                w = dict(logits=x, params=p, u=u, hist=hist, hist_len=length)
                assert np.array_equal(tokens, gpu_rows(ctx, w, hist_counts=counts)["tokens"]), (levels, penalised)
    finally:
        ctx.close()
