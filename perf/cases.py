"""Timing cases of the token-selection library: what a serving engine asks of it, over the sizes it is used at.

A case is a dict of plain values; "kind" says which public entry points one pass calls:

  sample    gse_sample over a resident batch (the C ABI of include/gse.h), as an engine's decode step calls it
  step      sampling.sample(), the drop-in Python surface, with a MaskBatch and a History; returns its list of tokens
  verify    gse_verify_tree over the draft trees of many requests (spec.VerifyCall.launch)
  strict    gse_dist then gse_mss: the strict speculative nodes of a step, dist + mss, through the C ABI
  node      sampling.dist() then spec.mss() at one strict node, the drop-in Python surface
  dist      gse_dist: the fp64 distributions of a batch
  pick      gse_draft_pick: a drafter level's children; with "q" also gse_qprob, the children's draft distributions

The inputs are drawn on the GPU from the seed. Logits laws: "normal" (flat rows), "zipf" (a normal plus a Zipf slope over
a random ranking of the tokens: what a trained model's rows look like) and "gumbel" (nucleus rows of a few hundred
tokens).
"""
import ctypes as C
import importlib
import math
import random

import numpy as np
import torch

ge = importlib.import_module("goethe-engine_amd")
lib, sampling, spec = ge._lib, ge.sampling, ge.spec

M64 = (1 << 64) - 1
SALT_DRAFT = 1 << 42
TREES = {  # parent of each drafted node (node 0: the anchor)
    "chain4": [0, 1, 2, 3],
    "chain7": [0, 1, 2, 3, 4, 5, 6],
    "pair": [0, 1, 2, 3, 0, 5, 6, 7],              # two chains of four from the anchor
    "wide": [0, 0, 0, 1, 1, 2, 4, 4, 5, 7],        # EAGLE-like: three kids at the anchor, then one or two
}


def listed():
    return [
        # one user's chat decode: a single row, nucleus sampling, the latency that the user waits for
        dict(name="chat_1", kind="sample", rows=1, vocab=128256, dtype="bf16", law="zipf", params="nucleus", hist=0,
             masks="none", logprobs=0),
        # a small batch with top-k, top-p and a repetition penalty
        dict(name="topk_8", kind="sample", rows=8, vocab=32000, dtype="f32", law="normal", params="topk", hist=64,
             masks="none", logprobs=0),
        # grammar-constrained greedy decoding (tool calls, JSON)
        dict(name="grammar_64", kind="sample", rows=64, vocab=128256, dtype="f32", law="normal", params="greedy",
             hist=0, masks="all", logprobs=0),
        # the headline batch: heterogeneous requests with every penalty, cut and a quarter of them under a grammar
        dict(name="full_256", kind="sample", rows=256, vocab=151936, dtype="f32", law="zipf", params="mixed", hist=2048,
             masks="quarter", logprobs=0),
        # the largest batch: nucleus sampling with the top-20 logprobs returned
        dict(name="logprobs_1024", kind="sample", rows=1024, vocab=262144, dtype="bf16", law="gumbel",
             params="nucleus", hist=0, masks="none", logprobs=20),
        # the same service through the Python drop-in, over an odd vocabulary
        dict(name="step_24", kind="step", rows=24, vocab=50257, dtype="f32", law="zipf", params="mixed", hist=333,
             masks="quarter", logprobs=0),
        # a verify round of a large speculative batch, rejection acceptance with the drafter's logits
        dict(name="verify_32", kind="verify", requests=32, tree="pair", vocab=128256, dtype="f32", accept="rejection",
             top_p=1.0),
        # a verify round of a few chats: one short chain each, bf16 logits, a nucleus at the target
        dict(name="verify_4", kind="verify", requests=4, tree="chain4", vocab=151936, dtype="bf16",
             accept="rejection", top_p=0.95),
        # strict nodes of a step (dist + mss) when the engine walks its trees itself
        dict(name="strict_16", kind="strict", rows=16, kids=2, vocab=128256, dtype="f32", law="zipf", top_p=0.95),
        # the same for one node, through Python
        dict(name="node_1", kind="node", rows=1, kids=2, vocab=50257, dtype="f32", law="zipf", top_p=1.0),
        # a drafter's level: four best children of each node of 16 sequences' beams
        dict(name="draft_greedy_64", kind="pick", rows=64, n=4, t=0.0, vocab=128256, dtype="bf16", q=False),
        # a sampling drafter's level with the draft distributions that rejection acceptance reads
        dict(name="draft_sampled_32", kind="pick", rows=32, n=2, t=0.8, vocab=32000, dtype="f32", q=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _vocab(rng, hi):
    """A vocabulary: a model's, or any size of the range (odd ones among them)."""
    v = [v for v in (32000, 50257, 128256, 151936, 262144) if v <= hi]
    return rng.choice(v) if v and rng.random() < 0.4 else _log_int(rng, min(4000, hi), hi)


def draw(rng):
    kind = rng.choice(["sample"] * 5 + ["step", "verify", "verify", "strict", "node", "dist", "pick", "pick"])
    dtype, law = rng.choice(["f32", "bf16"]), rng.choice(["zipf", "zipf", "normal", "gumbel"])
    if kind == "sample":
        rows = _log_int(rng, 1, 1024)
        v = _vocab(rng, min(262144, (1024 * 262144 if dtype == "bf16" else 512 * 262144) // rows))
        par = rng.choice(["greedy", "topk", "nucleus", "mixed"])
        return dict(kind=kind, rows=rows, vocab=v, dtype=dtype, law=law, params=par,
                    hist=rng.choice([0, _log_int(rng, 16, 2048)]), masks=rng.choice(["none", "none", "quarter", "all"]),
                    logprobs=rng.choice([0, 0, 5, 20]))
    if kind == "step":
        return dict(kind=kind, rows=_log_int(rng, 1, 64), vocab=_vocab(rng, 151936), dtype=dtype, law=law,
                    params=rng.choice(["greedy", "topk", "nucleus", "mixed"]), hist=_log_int(rng, 16, 1024),
                    masks=rng.choice(["none", "quarter", "all"]), logprobs=0)
    if kind == "verify":
        return dict(kind=kind, requests=_log_int(rng, 1, 32), tree=rng.choice(sorted(TREES)), vocab=_vocab(rng, 128256),
                    dtype=dtype, accept=rng.choice(["rejection", "rejection", "exact"]), top_p=rng.choice([1.0, 0.95]))
    if kind in ("strict", "node"):
        return dict(kind=kind, rows=_log_int(rng, 1, 64) if kind == "strict" else 1, kids=rng.randint(1, 4),
                    vocab=_vocab(rng, 151936), dtype=dtype, law=law, top_p=rng.choice([1.0, 0.95, 0.8]))
    if kind == "dist":
        return dict(kind=kind, rows=_log_int(rng, 1, 64), vocab=_vocab(rng, 262144), dtype=dtype, law=law,
                    top_p=rng.choice([1.0, 0.95, 0.8]))
    t = rng.choice([0.0, 0.6, 1.0])
    return dict(kind=kind, rows=_log_int(rng, 1, 128), n=rng.randint(1, 8), t=t, vocab=_vocab(rng, 151936), dtype=dtype,
                q=t > 0 and rng.random() < 0.5)


# ---- inputs ------------------------------------------------------------------------------------------------------------

def _dev():
    return torch.device("cuda", torch.cuda.current_device())


def _logits(g, rows, vocab, law, dtype, dev, want_ranks=False):
    """[rows, vocab] logits of the law, and for histories the token of each rank ([rows, vocab], zipf rows only)."""
    x = torch.randn((rows, vocab), generator=g, device=dev)
    by_rank = None
    if law == "zipf":
        by_rank = torch.argsort(torch.rand((rows, vocab), generator=g, device=dev), dim=1)
        slope = 1.1 * torch.log1p(torch.arange(vocab, device=dev, dtype=torch.float32))
        x = x.mul_(2.5).scatter_add_(1, by_rank, -slope.expand(rows, vocab))
        x -= x.mean(dim=1, keepdim=True)
    elif law == "gumbel":
        x = torch.rand((rows, vocab), generator=g, device=dev).clamp_(1e-9, 1 - 6e-8).log_().neg_().log_().mul_(-1.5)
    else:
        x.mul_(2.0)
    x = x.to(torch.bfloat16) if dtype == "bf16" else x
    return x, (by_rank if want_ranks else None)


def _params(case, rng):
    """One SamplingParams per row."""
    out = []
    lp = case.get("logprobs") or None
    for _ in range(case["rows"]):
        style = case["params"]
        pen = dict(repetition_penalty=1.1) if case["hist"] else {}
        if style == "greedy":
            p = dict(temperature=0.0)
        elif style == "topk":
            p = dict(temperature=0.8, top_k=40, top_p=0.95)
        elif style == "nucleus":
            p = dict(temperature=1.0 if lp else 0.7, top_p=0.9)
        else:
            p = dict(temperature=rng.uniform(0.5, 1.5), top_k=rng.choice([0, 20, 50, 200]),
                     top_p=rng.uniform(0.8, 1.0), min_p=rng.choice([0.0, 0.05]))
            pen = dict(repetition_penalty=rng.uniform(1.0, 1.3), frequency_penalty=rng.random(),
                       presence_penalty=rng.random())
        out.append(sampling.SamplingParams(logprobs=lp, **p, **pen))
    return out


def _hist_ids(g, case, by_rank, dev):
    """[rows, hist] ids: Zipf ranks through the row's ranking, or uniform ids."""
    rows, v, h = case["rows"], case["vocab"], case["hist"]
    u = torch.rand((rows, h), generator=g, device=dev, dtype=torch.float64)
    if by_rank is None:
        return (u * v).long().clamp_(max=v - 1).int()
    cdf = torch.arange(1, v + 1, device=dev, dtype=torch.float64).pow_(-1.2).cumsum(0)
    ranks = torch.searchsorted(cdf, u * cdf[-1], right=True).clamp_(max=v - 1)
    return by_rank.gather(1, ranks).int()


def _mask_words(g, case, dev):
    """(packed words [rows, ceil(vocab / 32)], masked rows): grammar rows allow 20 runs of tokens and 200 scattered ids,
    the other rows of a "quarter" batch allow everything."""
    rows, v = case["rows"], case["vocab"]
    if case["masks"] == "none":
        return None
    words = (v + 31) // 32
    b = torch.ones((rows, words * 32), dtype=torch.bool, device=dev)
    b[:, v:] = False
    strict = torch.arange(0, rows, 1 if case["masks"] == "all" else 4, device=dev)
    k = len(strict)
    m = torch.zeros((k, words * 32 + 1), dtype=torch.int32, device=dev)
    start = (torch.rand((k, 20), generator=g, device=dev) * max(1, v - 420)).long()
    end = torch.minimum(start + 200 + (torch.rand((k, 20), generator=g, device=dev) * 221).long(), torch.tensor(v, device=dev))
    one = torch.ones((k, 20), dtype=torch.int32, device=dev)
    m.scatter_add_(1, start, one).scatter_add_(1, end, -one)
    sub = m.cumsum(1)[:, :words * 32] > 0
    sub.scatter_(1, (torch.rand((k, 200), generator=g, device=dev) * v).long().clamp_(max=v - 1), True)
    b[strict] = sub
    w = (b.view(rows, words, 32).long() << torch.arange(32, device=dev)).sum(2)
    return torch.where(w >= 1 << 31, w - (1 << 32), w).int()


def _rows(params, seeds, idxs):
    """The gse_row records of the params (72 bytes each, include/gse.h)."""
    r = np.zeros(len(params), dtype=lib.ROW)
    for i, p in enumerate(params):
        r[i] = (np.float32(p.temperature), p.top_k, p.top_p, p.min_p, np.float32(p.repetition_penalty),
                np.float32(p.frequency_penalty), np.float32(p.presence_penalty), -1, seeds[i], idxs[i], 0, 0,
                p.logprobs or 0, 0)
    return r


def _batch(x, rows, mask=None, hist=None):
    """A gse_batch over resident tensors (all kept alive by the caller)."""
    b = lib.Batch()
    b.size, b.dtype = C.sizeof(lib.Batch), lib.BF16 if x.dtype == torch.bfloat16 else lib.F32
    b.rows, b.vocab, b.ld, b.logits = x.shape[0], x.shape[1], x.stride(0), x.data_ptr()
    b.params = rows.data_ptr()
    if mask is not None:
        b.mask, b.mask_ld = mask.data_ptr(), mask.stride(0)
    if hist is not None:
        b.hist = hist.data_ptr()
    b.stream = torch.cuda.current_stream(x.device).cuda_stream
    return b


def _softmax64(x, t):
    z = x.double() / t
    e = torch.exp(z - z.max(dim=-1, keepdim=True).values)
    return e / e.sum(dim=-1, keepdim=True)


def _draw_kids(g, q, n):
    """n tokens drawn from each row of q ([rows, vocab] fp64)."""
    c = q.cumsum(1)
    u = torch.rand((q.shape[0], n), generator=g, device=q.device, dtype=torch.float64) * c[:, -1:]
    return torch.searchsorted(c, u).clamp_(max=q.shape[1] - 1)


def prepare(case, seed):
    dev = _dev()
    g = torch.Generator(device=dev).manual_seed(seed & 0x7FFFFFFF)
    rng = random.Random(seed)
    return dict(sample=_prep_sample, step=_prep_step, verify=_prep_verify, strict=_prep_strict, node=_prep_node,
                dist=_prep_dist, pick=_prep_pick)[case["kind"]](case, g, rng, dev)


def _selection(case, g, rng, dev):
    """What the sampling kinds share: logits, per-row params, seeds, token indexes, histories and mask words."""
    n = case["rows"]
    x, by_rank = _logits(g, n, case["vocab"], case["law"], case["dtype"], dev, want_ranks=case["hist"] > 0)
    hist = _hist_ids(g, case, by_rank, dev) if case["hist"] else None
    seeds, idxs = [rng.getrandbits(64) for _ in range(n)], [rng.randrange(4096) for _ in range(n)]
    return x, _params(case, rng), seeds, idxs, hist, _mask_words(g, case, dev)


def _prep_sample(case, g, rng, dev):
    x, params, seeds, idxs, hist, mask = _selection(case, g, rng, dev)
    n = case["rows"]
    r = _rows(params, seeds, idxs)
    if hist is not None:
        r["hist_begin"] = np.arange(n) * case["hist"]
        r["hist_end"] = (np.arange(n) + 1) * case["hist"]
    if mask is not None:
        r["mask_row"] = np.arange(n)
    rows = torch.from_numpy(r.view(np.uint8)).to(dev)
    b = _batch(x, rows, mask, hist)
    if case["params"] == "greedy":
        b.flags = lib.BATCH_NO_SPLIT  # (what the header advises for batches of greedy rows)
    o = lib.Out()
    o.size = C.sizeof(lib.Out)
    tokens = torch.empty(n, dtype=torch.int32, device=dev)
    o.tokens = tokens.data_ptr()
    out = dict(tokens=tokens)
    if case["logprobs"]:
        k = case["logprobs"]
        out["ids"] = torch.empty((n, k), dtype=torch.int32, device=dev)
        out["logprobs"] = torch.empty((n, k), dtype=torch.float32, device=dev)
        o.logprob_ids, o.logprobs, o.logprobs_ld = out["ids"].data_ptr(), out["logprobs"].data_ptr(), k
    return dict(kind="sample", h=lib.handle(dev.index, n, case["vocab"]), b=b, o=o, out=out,
                keep=(x, rows, mask, hist), x=x, params=params, seeds=seeds, idxs=idxs, hist=hist, mask=mask)


def _prep_step(case, g, rng, dev):
    x, params, seeds, idxs, hist, mask = _selection(case, g, rng, dev)
    n = case["rows"]
    h = None
    if hist is not None:
        h = sampling.History(n, case["hist"] + 64, dev)
        for r in range(n):
            h.set(r, hist[r])
    mb = None
    if mask is not None:
        mb = ge.grammar.MaskBatch(n, case["vocab"])
        words = mask.cpu()
        for r in range(n):
            mb.set(r, words[r])
    return dict(kind="step", x=x, params=params, seeds=seeds, idxs=idxs, history=h, masks=mb, hist=hist, mask=mask)


def _prep_verify(case, g, rng, dev):
    parents = TREES[case["tree"]]
    n, v = len(parents) + 1, case["vocab"]
    kids = spec.kids_of(parents)
    reqs, keep = [], []
    tgt = torch.randn((case["requests"] * n, v), generator=g, device=dev).mul_(2.0)
    p = sampling.SamplingParams(temperature=1.0, accept=case["accept"], top_p=case["top_p"])
    cast = (lambda t: t.to(torch.bfloat16)) if case["dtype"] == "bf16" else (lambda t: t)
    for a in range(case["requests"]):
        drf = tgt[a * n:(a + 1) * n] + 0.5 * torch.randn((n, v), generator=g, device=dev)
        drf = cast(drf)
        inner = [u for u in range(n) if kids[u]]
        most = max(len(k) for k in kids)
        drawn = dict(zip(inner, _draw_kids(g, _softmax64(drf[inner], 1.0), most).tolist()))
        toks = [0] * (n - 1)
        for u in inner:
            for k, c in enumerate(kids[u]):
                toks[c - 1] = drawn[u][k]
        reqs.append(dict(tokens=toks, parents=list(parents), params=p, seed=rng.getrandbits(63), nout=rng.randrange(512),
                         draft=drf, draft_t=1.0))
        keep.append(drf)
    tgt = cast(tgt)
    for a, r in enumerate(reqs):
        r["target"] = tgt[a * n:(a + 1) * n]
    call = spec.VerifyCall(reqs)
    for t in (call.e_tok, call.e_node):  # (entries past a request's emitted tokens are not written)
        t.fill_(-1)
    return dict(kind="verify", call=call, keep=(tgt, keep))


def _strict_nodes(case, g, dev):
    """Target logits, the draft distributions (fp64 rows) and the kids drawn from them."""
    x, _ = _logits(g, case["rows"], case["vocab"], case["law"], case["dtype"], dev)
    q = _softmax64(x.float() + 0.5 * torch.randn(x.shape, generator=g, device=dev), 1.0)
    return x, q, _draw_kids(g, q, case["kids"])


def _prep_strict(case, g, rng, dev):
    n, v = case["rows"], case["vocab"]
    x, q, kids = _strict_nodes(case, g, dev)
    seeds, idxs = [rng.getrandbits(64) for _ in range(n)], [rng.randrange(4096) for _ in range(n)]
    p = sampling.SamplingParams(temperature=1.0, top_p=case["top_p"], accept="rejection")
    rows = torch.from_numpy(_rows([p] * n, seeds, idxs).view(np.uint8)).to(dev)
    b = _batch(x, rows)
    probs = torch.empty((n, v), dtype=torch.float64, device=dev)
    ktok = kids.int().contiguous()
    kq = torch.arange(n, device=dev, dtype=torch.int32)[:, None].expand(n, case["kids"]).contiguous()
    sd = torch.from_numpy(np.array(seeds, np.uint64).view(np.int64)).to(dev)
    ix = torch.tensor(idxs, dtype=torch.int64, device=dev)
    out = dict(token=torch.empty(n, dtype=torch.int32, device=dev), kid=torch.empty(n, dtype=torch.int32, device=dev))
    m = lib.MssBatch()
    m.size, m.nodes, m.vocab, m.max_kids = C.sizeof(lib.MssBatch), n, v, case["kids"]
    m.p, m.p_ld, m.q, m.q_ld = probs.data_ptr(), v, q.data_ptr(), v
    m.kid_tok, m.kid_q, m.seed, m.idx = ktok.data_ptr(), kq.data_ptr(), sd.data_ptr(), ix.data_ptr()
    m.out_token, m.out_kid, m.stream = out["token"].data_ptr(), out["kid"].data_ptr(), b.stream
    return dict(kind="strict", h=lib.handle(dev.index, n, v), b=b, probs=probs, m=m, out=out,
                keep=(x, q, rows, ktok, kq, sd, ix))


def _prep_node(case, g, rng, dev):
    x, q, kids = _strict_nodes(case, g, dev)
    p = sampling.SamplingParams(temperature=1.0, top_p=case["top_p"], accept="rejection")
    return dict(kind="node", x=x[0], p=p, kids=[(int(t), q[0]) for t in kids[0].tolist()], seed=rng.getrandbits(63),
                i=rng.randrange(4096))


def _prep_dist(case, g, rng, dev):
    n, v = case["rows"], case["vocab"]
    x, _ = _logits(g, n, v, case["law"], case["dtype"], dev)
    p = sampling.SamplingParams(temperature=0.9, top_p=case["top_p"])
    rows = torch.from_numpy(_rows([p] * n, [0] * n, [0] * n).view(np.uint8)).to(dev)
    return dict(kind="dist", h=lib.handle(dev.index, n, v), b=_batch(x, rows), x=x, params=[p] * n,
                probs=torch.empty((n, v), dtype=torch.float64, device=dev), keep=rows)


def _prep_pick(case, g, rng, dev):
    n, v, k = case["rows"], case["vocab"], case["n"]
    x, _ = _logits(g, n, v, "zipf", case["dtype"], dev)
    seeds, ats = [rng.getrandbits(63) for _ in range(n)], [rng.randrange(4096) for _ in range(n)]
    t = torch.full((n,), case["t"], dtype=torch.float64, device=dev)
    cnt = torch.full((n,), k, dtype=torch.int32, device=dev)
    sd, at = torch.tensor(seeds, device=dev), torch.tensor(ats, device=dev)
    out = dict(tokens=torch.empty((n, k), dtype=torch.int32, device=dev),
               logq=torch.empty((n, k), dtype=torch.float64, device=dev))
    b = lib.PickBatch()
    b.size, b.dtype = C.sizeof(lib.PickBatch), lib.BF16 if x.dtype == torch.bfloat16 else lib.F32
    b.rows, b.vocab, b.x, b.ld = n, v, x.data_ptr(), x.stride(0)
    b.temperature, b.n, b.seed, b.at = t.data_ptr(), cnt.data_ptr(), sd.data_ptr(), at.data_ptr()
    b.out_tokens, b.out_logq, b.out_ld = out["tokens"].data_ptr(), out["logq"].data_ptr(), k
    b.stream = torch.cuda.current_stream(dev).cuda_stream
    qr = None
    if case["q"]:
        out["q"] = torch.empty((n, v), dtype=torch.float64, device=dev)
        qr = lib.QRows()
        qr.size, qr.kind = C.sizeof(lib.QRows), lib.Q_LOGITS_BF16 if b.dtype == lib.BF16 else lib.Q_LOGITS_F32
        qr.rows, qr.q, qr.ld, qr.temperature = n, x.data_ptr(), x.stride(0), t.data_ptr()
    return dict(kind="pick", h=lib.handle(dev.index, n, v), b=b, qr=qr, out=out, x=x, seeds=seeds, ats=ats,
                keep=(t, cnt, sd, at))


# ---- one pass ------------------------------------------------------------------------------------------------------------

def run(s):
    kind = s["kind"]
    if kind == "sample":
        s["h"].call("gse_sample", C.byref(s["b"]), C.byref(s["o"]))
        return s["out"]
    if kind == "step":
        toks = sampling.sample(s["x"], s["params"], s["seeds"], s["idxs"], s["masks"], history=s["history"])
        return dict(tokens=np.array(toks, np.int64))
    if kind == "verify":
        c = s["call"]
        c.launch()
        return dict(len=c.e_len, tokens=c.e_tok, nodes=c.e_node, status=c.e_st)
    if kind == "strict":  # (gse_mss overwrites the distributions, its scratch)
        s["h"].call("gse_dist", C.byref(s["b"]), s["probs"].data_ptr(), s["probs"].stride(0))
        s["h"].call("gse_mss", C.byref(s["m"]))
        return s["out"]
    if kind == "node":
        p = sampling.dist(s["x"], s["p"])
        token, kid = spec.mss(p, s["kids"], s["seed"], s["i"])
        return dict(p=p, token=token, kid=-1 if kid is None else kid)
    if kind == "dist":
        s["h"].call("gse_dist", C.byref(s["b"]), s["probs"].data_ptr(), s["probs"].stride(0))
        return s["probs"]
    s["h"].call("gse_draft_pick", C.byref(s["b"]))
    if s["qr"] is not None:
        q = s["out"]["q"]
        s["h"].call("gse_qprob", C.byref(s["qr"]), q.shape[1], q.data_ptr(), q.stride(0), C.c_void_p(s["b"].stream))
    return s["out"]


def work(case):
    """Each input read once and each output written once; operations: the scale, exponential and sum of each logit."""
    v, es = case["vocab"], 2 if case["dtype"] == "bf16" else 4
    kind = case["kind"]
    if kind == "verify":
        parents = TREES[case["tree"]]
        rows = len(parents) + 1 + (len(set(parents)) if case["accept"] == "rejection" else 0)
        n = case["requests"] * rows * v
        return {"bytes": n * es, "flops": 4 * n}
    n = case["rows"] * v
    if kind in ("sample", "step"):
        b = n * es + 4 * case["rows"] * (1 + case["hist"] + 2 * case["logprobs"])
        if case["masks"] != "none":
            b += 4 * case["rows"] * ((v + 31) // 32)
        return {"bytes": b, "flops": (1 if case["params"] == "greedy" else 4) * n}
    if kind in ("strict", "node"):  # (the logits in, the draft rows in; the distributions out for "node")
        return {"bytes": n * (es + 8 + (8 if kind == "node" else 0)), "flops": 6 * n}
    if kind == "dist":
        return {"bytes": n * (es + 8), "flops": 5 * n}
    return {"bytes": n * (es + (8 if case["q"] else 0)), "flops": (4 if case["t"] > 0 else 1) * n}


def tolerance(case):
    """Tokens, kids and paths are the same. The numbers beside them are fp64 probabilities and log-probabilities (about
    an ulp per exponential and per sum), and fp32 roundings of fp64 log-probabilities (half an fp32 ulp)."""
    kind = case["kind"]
    if kind in ("node", "dist"):
        return {"rel": 4e-15, "max": 1e-14}
    if kind == "pick":
        return {"rel": 4e-15, "max": 1e-14} if case["t"] > 0 else "exact"
    if kind == "sample" and case["logprobs"]:
        return {"rel": 1e-7, "max": 2.4e-7}
    return "exact"


# ---- the same in plain torch, 64 bits ------------------------------------------------------------------------------------

def _mix(seed, i):
    z = (seed + (i + 1) * 0x9E3779B97F4A7C15) & M64
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & M64
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & M64
    return z ^ (z >> 31)


def _uniform(seed, i):
    return (_mix(seed, i) >> 11) / float(1 << 53)


def _processed(x, p, hist, mask):
    """One row's logits after the penalties and the mask; these are fp32 operations by definition."""
    v = x.shape[0]
    x = x.float().clone()
    if hist is not None:
        c = torch.bincount(hist.long(), minlength=v)
        f = lambda a: torch.tensor(a, dtype=torch.float32, device=x.device)  # noqa: E731
        y = torch.where(x < 0, x * f(p.repetition_penalty), x / f(p.repetition_penalty))
        y = y - f(p.frequency_penalty) * c.float()
        y = y - f(p.presence_penalty)
        x = torch.where(c > 0, y, x)
    if mask is not None:
        bit = (mask[:, None] >> torch.arange(32, device=x.device, dtype=torch.int32)) & 1
        x = torch.where(bit.reshape(-1)[:v].bool(), x, torch.tensor(-math.inf, device=x.device))
    return x


def _sorted_kept(x, p):
    """(order, z descending, exp(z - max), keep) of one sampled row: z = fp32(x / fp32(T)), the rest in 64 bits."""
    z = x / torch.tensor(p.temperature, dtype=torch.float32, device=x.device)
    zs, order = torch.sort(z, descending=True, stable=True)
    zs = zs.double()
    e = torch.exp(zs - zs[0])
    q = e / e.sum()
    keep = q.cumsum(0) - q < p.top_p
    if p.top_k:
        keep[p.top_k:] = False
    if p.min_p:
        keep &= q >= p.min_p * q[0]
    return order, zs, e, keep


def _exact_rows(s, case):
    """(tokens, top ids, top log-probabilities) of a sampling batch."""
    toks, ids, lps = [], [], []
    k = case["logprobs"]
    for r, p in enumerate(s["params"]):
        x = _processed(s["x"][r], p, None if s["hist"] is None else s["hist"][r],
                       None if s["mask"] is None else s["mask"][r])
        if p.temperature == 0:
            toks.append(int(x.argmax()))
            order = None
            if k:
                zs, order = torch.sort(x, descending=True, stable=True)
                zs = zs.double()
        else:
            order, zs, e, keep = _sorted_kept(x, p)
            c = (e * keep).cumsum(0)
            j = int((c < _uniform(s["seeds"][r], s["idxs"][r]) * c[-1]).sum())
            toks.append(int(order[max(min(j, int(keep.sum()) - 1), 0)]))
        if k:
            lse = torch.log(torch.exp(zs - zs[0]).sum())
            ids.append(order[:k])
            lps.append(zs[:k] - zs[0] - lse)
    return toks, ids, lps


def exact(case, seed):
    kind = case["kind"]
    if kind in ("verify", "strict"):  # (whole numbers only)
        return None
    s = prepare(case, seed)
    if kind == "sample":
        toks, ids, lps = _exact_rows(s, case)
        out = dict(tokens=torch.tensor(toks))
        if case["logprobs"]:
            out.update(ids=torch.stack(ids), logprobs=torch.stack(lps))
        return out
    if kind == "step":
        return dict(tokens=np.array(_exact_rows(s, case)[0], np.int64))
    if kind in ("node", "dist"):
        rows, params = (s["x"][None], [s["p"]]) if kind == "node" else (s["x"], s["params"])
        out = torch.zeros(rows.shape, dtype=torch.float64, device=rows.device)
        for r, p in enumerate(params):
            order, _, e, keep = _sorted_kept(rows[r].float(), p)
            e = e * keep
            out[r, order] = e / e.sum()
        return dict(p=out[0], token=None, kid=None) if kind == "node" else out
    x, t, k = s["x"].double(), case["t"], case["n"]
    if t == 0:
        v, order = torch.sort(x, dim=1, descending=True, stable=True)
        return dict(tokens=order[:, :k], logq=v[:, :k])
    q = _softmax64(x, t)
    z = x / t
    lq = z - torch.logsumexp(z, 1, keepdim=True)
    c = q.cumsum(1)
    u = torch.tensor([[_uniform(_mix(sd, SALT_DRAFT + j), at) for j in range(k)] for sd, at in zip(s["seeds"], s["ats"])],
                     dtype=torch.float64, device=x.device)
    toks = torch.searchsorted(c, u * c[:, -1:]).clamp_(max=x.shape[1] - 1)
    out = dict(tokens=toks, logq=lq.gather(1, toks))
    if case["q"]:
        out["q"] = q
    return out
