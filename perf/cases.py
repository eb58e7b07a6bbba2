"""The sampler's work as its users have it done: cases for timing, with their inputs and the call of each.

A case is a dict of plain values:
  rows, vocab   the batch; pad: elements between a row's end and the next row (logits_stride - vocab)
  logits        "spiked": N(0, 3^2) with up to 50 tokens raised by 10 in each row (a model that knows what comes next),
                "normal": N(0, 3^2), "stress": half the rows Student-t(3) * 4, half N(0, 0.1^2)
  params        what the rows ask for (row_params())
  hist          tokens of history in every row (Zipf over the vocabulary), 0: none; with the penalties 1.1 / 0.2 / 0.3
  mask          share of the vocabulary that a row's mask allows, 0: no mask
  draft         speculative verification: a draft token and a second uniform for every row
  scores        the candidates' number, the total and the token's weight are wanted too (an API's logprobs)
  call          "hinted": device pointers and the host copy of the parameters; "plain": device pointers alone;
                "static": the call on the library's own scratch memory; "host": the call on host pointers

Outputs are whole numbers and the fp32 values of a defined sequence of operations: they do not depend on the
implementation, so every case is compared exactly.
"""
import ctypes
import math

import numpy as np
import torch

from mako_amd import api, workloads

KINDS = ("greedy", "top_k", "nucleus", "serving", "temperature", "min_p", "top_k_alone", "wide_top_k", "any")
MAX_ELEMENTS = 512 * workloads.V_DEEPSEEK  # of the largest batch


def case(name, rows, vocab, params, logits="spiked", pad=0, hist=0, mask=0.0, draft=False, scores=False, call="hinted"):
    return dict(name=name, rows=rows, vocab=vocab, pad=pad, logits=logits, params=params, hist=hist, mask=mask,
                draft=draft, scores=scores, call=call)


def listed():
    small, large = workloads.V_DEEPSEEK, workloads.V_LARGE
    return [
        # one sequence on its own, as a chat on one's own machine: latency is all that counts
        case("greedy_1", 1, large, "greedy", "normal", hist=512),
        case("top_k_1", 1, small, "top_k"),
        case("nucleus_1", 1, large, "nucleus", "normal", hist=512, scores=True),
        # the C++ class mako::gen::Sampler: one row of host logits, its history as (token, count) pairs
        case("host_1", 1, small, "top_k", hist=256, call="host"),
        # a small model in a decode loop that must not allocate
        case("static_8", 8, 32000, "serving", hist=512, call="static"),
        # a vocabulary that is a multiple of nothing, all kinds of requests in one batch, and a caller that keeps the
        # parameters on the device only
        case("ragged_24", 24, 151553, "any", "normal", hist=300, call="plain"),
        # the decode batch of a server
        case("decode_64", 64, small, "serving", hist=2048),
        # requests that set neither top_k nor top_p, and requests that set top_k alone
        case("temperature_64", 64, small, "temperature", scores=True),
        case("top_k_alone_64", 64, small, "top_k_alone"),
        # 32 sequences, eight positions each, verified against drafts under a grammar's masks
        case("verify_256", 256, small, "top_k", "spiked", mask=0.5, draft=True),
        # full-vocabulary cutoffs, on rows as peaked and as flat as they come
        case("nucleus_256", 256, large, "nucleus", "stress"),
        # the largest decode batch
        case("decode_512", 512, small, "serving", hist=1024, scores=True),
    ]


def _spread(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    call = rng.choice(("hinted",) * 6 + ("plain", "plain", "static", "host"))
    params = rng.choice(KINDS)
    vocab = _spread(rng, 8000, 160000)
    if rng.random() < 0.6:  # most vocabularies are padded to a multiple of 64; the others are as they come
        vocab = (vocab + 63) // 64 * 64
    if call == "static":
        vocab = min(vocab, api.STATIC_MAX_VOCAB)
    most = {"static": api.STATIC_MAX_ROWS, "host": 16}.get(call, 512)
    if params == "nucleus":
        most = min(most, 256)
    elif params in ("top_k_alone", "wide_top_k", "any") or (call == "plain" and params in ("temperature", "min_p")):
        most = min(most, 64)
    rows = _spread(rng, 1, max(1, min(most, MAX_ELEMENTS // vocab)))
    return dict(rows=rows, vocab=vocab, pad=rng.choice((0, 0, 0, 64, 1)) if call != "host" else 0,
                logits=rng.choice(("spiked", "spiked", "normal", "stress")), params=params,
                hist=rng.choice((0, _spread(rng, 16, 4096))), mask=rng.choice((0.0, 0.0, 0.01, 0.5, 0.9)),
                draft=rng.random() < 0.2, scores=call != "host" and rng.random() < 0.3, call=call)


def row_params(kind, rows, rng, penalised):
    """The rows' sampling parameters: PARAMS_DTYPE[rows]."""
    p = api.make_params(rows)
    if penalised:
        p["repetition_penalty"], p["frequency_penalty"], p["presence_penalty"] = 1.1, 0.2, 0.3
    if kind == "greedy":
        p["temperature"] = 0.0
    elif kind == "top_k":
        p["temperature"], p["top_k"], p["top_p"] = (0.7, 40, 0.95)
    elif kind == "nucleus":
        p["top_p"] = 0.9
    elif kind == "serving":  # a server's decode batch: every request has its own
        p["temperature"] = rng.uniform(0.3, 1.2, rows)
        p["top_k"] = rng.choice([0, 20, 50, 100], rows)
        p["top_p"] = np.minimum(rng.uniform(0.8, 1.0, rows).astype(np.float32), np.float32(1.0 - 2.0**-24))
    elif kind == "temperature":
        p["temperature"] = rng.uniform(0.5, 1.2, rows)
    elif kind == "min_p":
        p["temperature"], p["min_p"] = 1.0, rng.choice([0.02, 0.05, 0.1], rows)
    elif kind == "top_k_alone":
        p["temperature"], p["top_k"] = 0.7, 40
    elif kind == "wide_top_k":
        p["temperature"], p["top_k"], p["top_p"] = 1.0, rng.choice([200, 500, 1000], rows), 0.95
    elif kind == "any":  # each row one of the kinds
        parts = [row_params(k, rows, rng, penalised) for k in KINDS[:-1]]
        which = rng.permutation(np.arange(rows) % len(parts))
        for k, part in enumerate(parts):
            p[which == k] = part[which == k]
    else:
        raise ValueError(kind)
    return p


def row_logits(kind, rows, vocab, stride, gen):
    """fp32 [rows, stride] on the GPU."""
    x = torch.randn(rows, stride, generator=gen, device="cuda")
    if kind == "stress":
        half = rows // 2
        if half:
            z = torch.randn(3, half, stride, generator=gen, device="cuda")
            x[:half] *= 4.0 / (z.square_().sum(0) / 3.0).sqrt_()
        x[half:] *= 0.1
        return x
    x *= 3.0
    if kind == "spiked":
        at = torch.randint(0, vocab, (rows, 50), generator=gen, device="cuda")
        n = torch.randint(1, 51, (rows, 1), generator=gen, device="cuda")
        x.scatter_add_(1, at, torch.where(torch.arange(50, device="cuda") < n, 10.0, 0.0))
    return x


def row_history(rows, vocab, length, gen):
    """int32 [rows, length]: token k - 1 with probability proportional to k^-1.1."""
    cdf = torch.arange(1, vocab + 1, dtype=torch.float64, device="cuda").pow_(-1.1).cumsum_(0)
    r = torch.rand(rows, length, dtype=torch.float64, generator=gen, device="cuda") * cdf[-1]
    return torch.searchsorted(cdf, r).clamp_(max=vocab - 1).to(torch.int32)


def row_masks(rows, vocab, share, gen):
    """uint32 words as int32 [rows, ceil(vocab / 32)]: bit i & 31 of word i >> 5 allows token i."""
    words = (vocab + 31) // 32
    bits = torch.rand(rows, words * 32, generator=gen, device="cuda") < share
    bits[:, vocab:] = False
    bits[:, 0] = True  # (no mask clears every token)
    weight = (1 << torch.arange(32, device="cuda")).to(torch.int64)
    out = torch.empty(rows, words, dtype=torch.int32, device="cuda")
    for r in range(0, rows, 64):
        v = (bits[r:r + 64].view(-1, words, 32) * weight).sum(2)
        out[r:r + 64] = torch.where(v >= 1 << 31, v - (1 << 32), v).to(torch.int32)
    return out


_contexts = {}  # the one in use: a program keeps its context for all its batches


def context(rows, vocab, hist):
    key = (rows, vocab, hist)
    if key not in _contexts:
        _contexts.clear()
        _contexts[key] = api.SamplerContext(max_rows=rows, max_vocab=vocab, max_hist=hist)
    return _contexts[key]


def prepare(c, seed):
    rows, vocab = c["rows"], c["vocab"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rng = np.random.Generator(np.random.PCG64([seed, 7]))
    logits = row_logits(c["logits"], rows, vocab, vocab + c["pad"], gen)
    params = row_params(c["params"], rows, rng, c["hist"] > 0)
    t = dict(logits=logits, params=torch.from_numpy(params.view(np.uint8).copy()).cuda(),
             u=torch.rand(rows, generator=gen, device="cuda"))
    if c["hist"]:
        t["hist"] = row_history(rows, vocab, c["hist"], gen)
        t["hist_len"] = torch.full((rows,), c["hist"], dtype=torch.int32, device="cuda")
    if c["mask"]:
        t["mask"] = row_masks(rows, vocab, c["mask"], gen)
    if c["draft"]:  # most drafts are the model's own favourite, the others some token
        best = logits[:, :vocab].argmax(1).to(torch.int32)
        other = torch.randint(0, vocab, (rows,), generator=gen, device="cuda", dtype=torch.int32)
        t["draft"] = torch.where(torch.rand(rows, generator=gen, device="cuda") < 0.7, best, other)
        t["u2"] = torch.rand(rows, generator=gen, device="cuda")
    ctx = context(rows, vocab, c["hist"])
    out = dict(tokens=torch.zeros(rows, dtype=torch.int32, device="cuda"))
    if c["draft"]:
        out["accepted"] = torch.zeros(rows, dtype=torch.uint8, device="cuda")
    if c["scores"]:
        out["n_cand"] = torch.zeros(rows, dtype=torch.int32, device="cuda")
        out["total"] = torch.zeros(rows, device="cuda")
        out["q"] = torch.zeros(rows, device="cuda")
    if c["call"] == "host":
        return prepare_host(c, ctx, t, params)
    d = api.Desc()
    d.logits, d.logits_stride, d.n_rows, d.n_vocab = logits.data_ptr(), vocab + c["pad"], rows, vocab
    d.params, d.u = t["params"].data_ptr(), t["u"].data_ptr()
    if c["hist"]:
        d.hist_tokens, d.hist_stride, d.hist_len = t["hist"].data_ptr(), c["hist"], t["hist_len"].data_ptr()
    if c["mask"]:
        d.mask, d.mask_stride = t["mask"].data_ptr(), t["mask"].shape[1]
    if c["draft"]:
        d.draft, d.u2, d.out_accepted = t["draft"].data_ptr(), t["u2"].data_ptr(), out["accepted"].data_ptr()
    d.out_tokens = out["tokens"].data_ptr()
    if c["scores"]:
        d.out_n_cand, d.out_total, d.out_q = (out[k].data_ptr() for k in ("n_cand", "total", "q"))
    return dict(call=c["call"], ctx=ctx, desc=d, out=out, keep=t, params=params,
                params_host=params.ctypes.data if c["call"] == "hinted" else None)


def prepare_host(c, ctx, t, params):
    """The same inputs in host memory, the histories as (token, count) pairs, and the arguments of the host call."""
    rows, vocab = c["rows"], c["vocab"]
    h = dict(logits=t["logits"].cpu().numpy(), params=params, u=t["u"].cpu().numpy(), tokens=np.zeros(rows, np.int32))
    if c["hist"]:
        pairs = [np.unique(r, return_counts=True) for r in t["hist"].cpu().numpy()]
        longest = max(len(ids) for ids, _ in pairs)
        h["ids"], h["counts"] = np.zeros((rows, longest), np.int32), np.zeros((rows, longest), np.uint32)
        h["len"] = np.array([len(ids) for ids, _ in pairs], np.uint32)
        for r, (ids, counts) in enumerate(pairs):
            h["ids"][r, :len(ids)], h["counts"][r, :len(ids)] = ids, counts
    if c["mask"]:
        h["mask"] = t["mask"].cpu().numpy()
    out = dict(tokens=h["tokens"])
    if c["draft"]:
        h["draft"], h["u2"] = t["draft"].cpu().numpy(), t["u2"].cpu().numpy()
        out["accepted"] = h["accepted"] = np.zeros(rows, np.uint8)

    def at(k):
        return ctypes.c_void_p(h[k].ctypes.data) if k in h else None

    args = (ctypes.c_void_p(ctx.ptr), at("logits"), vocab, rows, vocab, at("params"), at("u"), at("mask"),
            h["mask"].shape[1] if c["mask"] else 0, at("ids"), at("counts"), h["ids"].shape[1] if c["hist"] else 0,
            at("len"), at("draft"), at("u2"), at("accepted"), at("tokens"))
    return dict(call="host", ctx=ctx, args=args, out=out, keep=h)


def run(s):
    if s["call"] == "host":
        rc = s["ctx"].lib.mako_sampler_sample_host(*s["args"])
        if rc != api.MAKO_OK:
            raise api.MakoError("mako_sampler_sample_host: %d %s" % (rc, s["ctx"].last_error()))
    elif s["call"] == "static":
        s["ctx"].sample_batch_static(s["desc"])
    else:
        s["ctx"].sample_batch(s["desc"], params_host=s["params_host"])
    return s["out"]


def work(c):
    """Each input read once and each output written once; an operation or two per logit (the kernels are no contractions)."""
    row = 4 * c["vocab"] + 28 + 4 + 4 + 4 * c["hist"]
    if c["mask"]:
        row += 4 * ((c["vocab"] + 31) // 32)
    if c["draft"]:
        row += 4 + 4 + 1
    if c["scores"]:
        row += 12
    return dict(bytes=c["rows"] * row, flops=2 * c["rows"] * c["vocab"])


def tolerance(c):
    return "exact"
