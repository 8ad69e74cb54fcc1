"""GPU parity of the row passes (draw, mss, pick) at the edges of their slices and segments, against the oracle: tokens and
accepted kids are compared exactly (a draw within rounding of a prefix boundary has a probability of about 1e-13)."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import sampling_ref as ora
from oracle import spec_ref as spo

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 63, 64, 65, 4095, 4096, 4097, 50257, 262147]


@pytest.mark.parametrize("v", SIZES)
def test_draw_sizes(ge, gpu, v):
    """Positive rows, sparse rows (long zero runs before, between and after the mass) and u at 0 and just below 1."""
    rng = np.random.default_rng(v)
    for kind in range(3):
        q = rng.random(v)
        if kind == 1:
            q[rng.random(v) < 0.999] = 0.0
            q[rng.integers(0, v)] = 0.5
        if kind == 2:
            q[:] = 0.0
            q[v // 2] = 1.0
        qt = torch.from_numpy(q).to(gpu)
        for u in [0.0, 0.3, 0.9, 1.0 - 2.0 ** -53]:
            assert ge.sampling.draw(qt, u) == ora.draw(q, u), (v, kind, u)
    with pytest.raises(IndexError):
        ge.sampling.draw(torch.zeros(v, dtype=torch.float64, device=gpu), 0.5)


def test_draw_never_takes_a_zero(ge, gpu):
    """Rows with long runs of zeros, u at the prefix of a random token and the doubles next to it: the slices, segments
    and tokens are summed in different orders, and whichever of them rounds to the threshold first, the drawn token has
    a positive weight and its exact prefix lies within rounding of u (sums of 9001 terms: 1e-13)."""
    lib = ge._lib
    v, rows = 9001, 6000
    rng = np.random.default_rng(12)
    q = rng.random((20, v)) * (rng.random((20, v)) < 0.02)
    q[:, 4090:4200] = 0.0
    c = q.cumsum(1)
    src = np.arange(rows) % 20
    at = np.array([rng.choice(np.nonzero(q[r])[0]) for r in src])
    u = c[src, at] / c[src, -1] + rng.integers(-6, 7, rows) * 2.0 ** -53
    u = np.clip(u, 2.0 ** -53, 1.0 - 2.0 ** -53)
    qd = torch.from_numpy(q).to(gpu)[torch.from_numpy(src).to(gpu)].contiguous()
    ud = torch.from_numpy(u).to(gpu)
    out = torch.full((rows,), -7, dtype=torch.int32, device=gpu)
    h = lib.handle(gpu.index, 64, v)
    h.call("gse_draw", qd.data_ptr(), v, rows, v, ud.data_ptr(), out.data_ptr(), lib.stream_of(gpu.index))
    t = out.cpu().numpy()
    assert (t >= 0).all() and (q[src, t] > 0).all(), t[q[src, t] <= 0]
    lo, hi = (c[src, t] - q[src, t]) / c[src, -1], c[src, t] / c[src, -1]
    assert (u >= lo - 1e-13).all() and (u <= hi + 1e-13).all()


def _nodes(v, n, rng):
    """Nodes of 0 .. 5 kids over [n, v] targets: kids with a distribution of their own, kids sharing one, one-hot kids;
    the kids' tokens are where q most exceeds p, so that most are rejected and the deeper levels run."""
    p = rng.random((n, v)) ** 4
    p[:, rng.random(v) < 0.3] = 0.0
    p[:, 0] += 1e-3
    p /= p.sum(1, keepdims=True)
    kids = []
    for a in range(n):
        q = [rng.random(v) ** 4 for _ in range(2)]
        q = [x / x.sum() for x in q]
        ks = []
        for r in range(a % 6):
            if (a + r) % 4 == 3:
                ks.append((int(rng.integers(0, v)), None))
            else:
                j = (a + r) % 2
                ks.append((int(np.argsort(p[a] - q[j])[min(r, v - 1)]), q[j]))
        kids.append(ks)
    return p, kids


@pytest.mark.parametrize("v", SIZES)
def test_mss_sizes(ge, gpu, v):
    n = 12 if v < 100000 else 6
    p, kids = _nodes(v, n, np.random.default_rng(v))
    levels = set()
    for seed in range(3):
        toks, ks = ge.spec.mss_batch(torch.from_numpy(p).to(gpu), kids, [seed * 100 + a for a in range(n)], [5] * n)
        for a in range(n):
            want = spo.mss(p[a], kids[a], seed * 100 + a, 5)
            assert (toks[a], ks[a]) == want, (v, seed, a)
            levels.add(len(kids[a]) if want[1] is None else want[1])
    if v >= 63:
        assert max(levels) == 5, levels  # a node whose five kids were all rejected


@pytest.mark.parametrize("v", [200, 5000, 50257])
def test_mss_kids_past_the_sliced_levels(ge, gpu, v):
    """Nodes whose first three kids are rejected for certain (tokens of probability 0) and whose fourth is a coin flip on
    a token that each wave's first pass over the row writes: every wave must have read its probability by then. Tokens
    and kids against the oracle, and nothing but the oracle's answer over repeated calls."""
    n = 48
    rng = np.random.default_rng(v)
    p = rng.random((n, v)) ** 2
    p[:, [3, 70, 150]] = 0.0
    p /= p.sum(1, keepdims=True)
    kids = []
    for a in range(n):
        x = int([0, 1, 63, 64, 100, 128, 190, 199][a % 8])
        q = rng.random((3, v)) ** 2
        q[:, x] = 0.0
        q[:, [3, 70, 150]] += 0.1
        q = q / q.sum(1, keepdims=True)
        last = np.zeros(v)
        last[x] = 2.0 * p[a, x]  # (the residuals so far only raise p[x]: accepted with probability a half or more)
        last[(x + 1) % v] += 1.0 - last[x]
        kids.append([(3, q[0]), (70, q[1]), (150, q[2]), (x, last if a % 3 else None), (3, q[0]), (x, q[1])])
    pd = torch.from_numpy(p).to(gpu)
    want = [spo.mss(p[a], kids[a], a, 9) for a in range(n)]
    assert {r for _, r in want} >= {3, None}
    for _ in range(3):
        toks, ks = ge.spec.mss_batch(pd, kids, list(range(n)), [9] * n)
        assert list(zip(toks, ks)) == want


def test_rows_past_the_handles_size(ge, gpu):
    """A handle opened for one row of 64 tokens serves draw and mss over more rows of a longer vocabulary: its few
    slices widen and the rows go out in several launches."""
    lib = ge._lib
    h = lib.Handle(gpu.index, 1, 64)
    rng = np.random.default_rng(3)
    v, rows = 50257, 5
    q = rng.random((rows, v)) * (rng.random((rows, v)) < 0.5)
    u = rng.random(rows)
    qd, ud = torch.from_numpy(q).to(gpu), torch.from_numpy(u).to(gpu)
    out = torch.full((rows,), -7, dtype=torch.int32, device=gpu)
    for _ in range(2):
        h.call("gse_draw", qd.data_ptr(), v, rows, v, ud.data_ptr(), out.data_ptr(), lib.stream_of(gpu.index))
        assert out.cpu().tolist() == [ora.draw(q[r], u[r]) for r in range(rows)]
    p, kids = _nodes(v, 6, rng)
    kmax = 5
    kt, kq, qs = np.full((6, kmax), -1, np.int32), np.full((6, kmax), -1, np.int32), []
    for a, ks in enumerate(kids):
        for r, (x, qq) in enumerate(ks):
            kt[a, r] = x
            if qq is not None:
                kq[a, r] = len(qs)
                qs.append(qq)
    dev = lambda x: torch.from_numpy(np.ascontiguousarray(x)).to(gpu)  # noqa: E731
    pd, qd, ktd, kqd = dev(p), dev(np.stack(qs)), dev(kt), dev(kq)
    sd, ix = dev(np.arange(6, dtype=np.int64) + 40), dev(np.full(6, 9, np.int64))
    ot, ok = torch.empty(6, dtype=torch.int32, device=gpu), torch.empty(6, dtype=torch.int32, device=gpu)
    b = lib.MssBatch()
    b.size, b.nodes, b.vocab, b.max_kids = C.sizeof(lib.MssBatch), 6, v, kmax
    b.p, b.p_ld, b.q, b.q_ld = pd.data_ptr(), v, qd.data_ptr(), v
    b.kid_tok, b.kid_q, b.seed, b.idx = ktd.data_ptr(), kqd.data_ptr(), sd.data_ptr(), ix.data_ptr()
    b.out_token, b.out_kid = ot.data_ptr(), ok.data_ptr()
    b.stream = torch.cuda.current_stream(gpu).cuda_stream
    h.call("gse_mss", C.byref(b))
    want = [spo.mss(p[a], kids[a], 40 + a, 9) for a in range(6)]
    assert ot.cpu().tolist() == [t for t, _ in want]
    assert ok.cpu().tolist() == [-1 if r is None else r for _, r in want]
    h.close()


def test_two_streams_with_a_handle_each(ge, gpu):
    """draw, mss and qprob keep their partial sums in the handle's workspace: calls that overlap on two streams, each with
    its own handle (which the Python layer keeps per stream), do not disturb each other."""
    v, n = 128256, 8
    rng = np.random.default_rng(5)
    streams = [torch.cuda.Stream(gpu) for _ in range(2)]
    data = []
    for s in range(2):
        q, u = rng.random((n, v)), rng.random(n)
        p, kids = _nodes(v, n, rng)
        x = torch.from_numpy(rng.normal(size=(n, v)).astype(np.float32))
        want = ([ora.draw(q[r], u[r]) for r in range(n)], [spo.mss(p[a], kids[a], a, s) for a in range(n)])
        data.append((torch.from_numpy(q).to(gpu), torch.from_numpy(u).to(gpu), torch.from_numpy(p).to(gpu), kids,
                     x.to(gpu), torch.softmax(x.double() / 0.7, 1).numpy(), want))
    torch.cuda.synchronize()
    lib = ge._lib
    for _ in range(3):
        outs = []
        for s in range(2):
            with torch.cuda.stream(streams[s]):
                q, u, p, kids, x, _, _ = data[s]
                h = lib.handle(gpu.index, n, v)
                out = torch.full((6, n), -7, dtype=torch.int32, device=gpu)
                for k in range(6):
                    h.call("gse_draw", q.data_ptr(), v, n, v, u.data_ptr(), out[k].data_ptr(), lib.stream_of(gpu.index))
                outs.append((h, out, ge.spec.qprob(x, 0.7)))
        assert outs[0][0] is not outs[1][0]
        for s in range(2):
            with torch.cuda.stream(streams[s]):
                _, _, p, kids, _, sm, want = data[s]
                toks, ks = ge.spec.mss_batch(p, kids, list(range(n)), [s] * n)
                assert list(zip(toks, ks)) == want[1]
                assert outs[s][1].cpu().tolist() == [want[0]] * 6
                np.testing.assert_allclose(outs[s][2].cpu().numpy(), sm, rtol=1e-13)


def test_rows_of_nearly_2_31_tokens(ge, gpu):
    """The last slice of a row of 2^31 - 1 tokens reaches past 2^31: draw and qprob read and write inside the row, and a
    longer row is refused."""
    lib = ge._lib
    v = 2 ** 31 - 1
    q = torch.zeros(v, dtype=torch.float64, device=gpu)
    q[5] = q[v - 1] = 1.0
    h = lib.Handle(gpu.index, 64, 64)
    st = lib.stream_of(gpu.index)
    out = torch.zeros(1, dtype=torch.int32, device=gpu)
    for u, want in ((0.3, 5), (0.7, v - 1)):
        ut = torch.tensor([u], dtype=torch.float64, device=gpu)
        h.call("gse_draw", q.data_ptr(), v, 1, v, ut.data_ptr(), out.data_ptr(), st)
        assert out.item() == want
    x = torch.full((1, v), -float("inf"), dtype=torch.bfloat16, device=gpu)
    x[0, 3] = x[0, v - 1] = 2.0
    t = torch.ones(1, dtype=torch.float64, device=gpu)
    r = lib.QRows()
    r.size, r.kind = C.sizeof(lib.QRows), lib.Q_LOGITS_BF16
    r.rows, r.q, r.ld, r.temperature = 1, x.data_ptr(), v, t.data_ptr()
    h.call("gse_qprob", C.byref(r), v, q.data_ptr(), v, st)
    assert q[3].item() == 0.5 and q[v - 1].item() == 0.5 and torch.count_nonzero(q).item() == 2
    with pytest.raises(RuntimeError, match="2\\^31"):
        h.call("gse_draw", q.data_ptr(), v + 1, 1, v + 1, t.data_ptr(), out.data_ptr(), st)
    r.ld = v + 1
    with pytest.raises(RuntimeError, match="2\\^31"):
        h.call("gse_qprob", C.byref(r), v + 1, q.data_ptr(), v + 1, st)
    m = lib.MssBatch()
    m.size, m.nodes, m.vocab, m.max_kids = C.sizeof(lib.MssBatch), 1, v + 1, 1
    m.p, m.p_ld = q.data_ptr(), v + 1
    m.kid_tok = m.kid_q = m.seed = m.idx = m.out_token = m.out_kid = out.data_ptr()
    with pytest.raises(RuntimeError, match="2\\^31"):
        h.call("gse_mss", C.byref(m))
    h.close()


def _pick_rows(v, rng):
    """Rows with ties everywhere (one value; two values), with the best tokens side by side, with -inf in most places,
    with a single finite token, and plain ones."""
    x = rng.normal(0, 3, size=(7, v)).astype(np.float32)
    x[1] = 0.25
    x[2] = (rng.random(v) < 0.5).astype(np.float32)
    x[3, v // 2:v // 2 + 20] += 30.0
    x[4, rng.random(v) < 0.99] = -np.inf
    x[4, -1] = 1.0
    x[5] = -np.inf
    x[5, v // 3] = -2.0
    return x


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("v", [1, 5, 64, 255, 4095, 4096, 4097, 50257, 262147])
def test_pick_sizes(ge, gpu, v, shift, dtype):
    """n best and n draws (n to 16) over whole and ragged slices, rows on and off a 16-byte boundary, t == 0 and t > 0
    rows in one call."""
    rng = np.random.default_rng(v + shift)
    x = torch.from_numpy(_pick_rows(v, rng))
    x = x.bfloat16() if dtype == "bf16" else x
    x32 = x.float().numpy()
    rows = len(x)
    buf = torch.zeros((rows, v + 3), dtype=x.dtype)
    buf[:, shift:shift + v] = x
    xd = buf.to(gpu)[:, shift:shift + v] if v > 1 else x.to(gpu)
    for t in ([0.0] * rows, [0.7] * rows, [0.0, 1.0, 1.0, 0.0, 2.5, 0.5, 1.0]):
        n = [min(v, k) for k in (16, 1, 7, 16, 3, 1, 4)]
        if t[4] == 0.0:  # (as many as there are tokens above -inf: the oracle then has no tie to break past them)
            n[4] = min(3, int((x32[4] > -np.inf).sum()))
        seeds, ats = [1000 + r for r in range(rows)], [3 * r for r in range(rows)]
        toks, vals = ge.spec.pick_batch(xd, n, t, seeds, ats)
        toks, vals = toks.cpu().numpy(), vals.cpu().numpy()
        for r in range(rows):
            want = spo.pick(x32[r], n[r], t[r], seeds[r], ats[r])
            assert list(toks[r, :n[r]]) == [w[0] for w in want], (v, t[r], r)
            np.testing.assert_allclose(vals[r, :n[r]], [w[2] for w in want], rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_pick_more_slices_than_the_device_holds(ge, gpu, dtype):
    """300 rows of five slices (the last one of five tokens): the workgroups take four slices each, ties and all, and the
    draws' values are those of the same rows alone."""
    rng = np.random.default_rng(17)
    v, rows = 4 * 4096 + 5, 301
    x = torch.from_numpy(np.concatenate([_pick_rows(v, rng) for _ in range(43)]))
    x = x.bfloat16() if dtype == "bf16" else x
    x32, xd = x.float().numpy(), x.to(gpu)
    n = [int(k) for k in rng.integers(1, 17, size=rows)]
    t = [float(k) for k in rng.choice([0.0, 0.0, 0.6, 1.0], size=rows)]
    seeds, ats = list(range(rows)), [7] * rows
    for r in range(rows):
        if t[r] == 0.0 and r % 7 in (4, 5):
            n[r] = min(n[r], int((x32[r] > -np.inf).sum()))
    toks, vals = ge.spec.pick_batch(xd, n, t, seeds, ats)
    toks, vals = toks.cpu().numpy(), vals.cpu().numpy()
    for r in range(rows):
        want = spo.pick(x32[r], n[r], t[r], seeds[r], ats[r])
        assert list(toks[r, :n[r]]) == [w[0] for w in want], (t[r], r)
        np.testing.assert_allclose(vals[r, :n[r]], [w[2] for w in want], rtol=1e-12, atol=1e-12)
    some = list(range(0, rows, 20))
    t1, v1 = ge.spec.pick_batch(xd[some], [n[r] for r in some], [t[r] for r in some], some, [7] * len(some))
    t1, v1 = t1.cpu().numpy(), v1.cpu().numpy()
    for i, r in enumerate(some):
        assert list(t1[i, :n[r]]) == list(toks[r, :n[r]]) and np.array_equal(v1[i, :n[r]], vals[r, :n[r]])


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("v", [1, 4095, 4097, 50257])
def test_qprob_sizes(ge, gpu, v, dtype):
    """Softmax rows over whole and ragged slices, on and off a 16-byte boundary, with -inf, masses far below the row's
    maximum, and the rows that are NaN everywhere (a NaN, a +inf, nothing above -inf); and the same through a handle whose
    few slices widen. q = exp(z - M) / E: each of z, the exponential, the sum and the quotient rounds within an ulp or two,
    and z's rounding (|z| 2^-53) is an error of the exponent, so 1e-13 covers |z| up to a few hundred."""
    rng = np.random.default_rng(v)
    x = torch.from_numpy(np.concatenate([_pick_rows(v, rng), np.full((3, v), 1.5, np.float32)]))
    x[0, 0] = -700.0
    x[7, v // 2] = np.nan
    x[8, v - 1] = np.inf
    x[9] = -np.inf
    x = x.bfloat16() if dtype == "bf16" else x
    x64 = x.double().numpy()
    t = [1.0, 0.5, 1.7, 2.0, 0.9, 1.0, 0.3, 1.0, 0.7, 1.0]
    buf = torch.zeros((len(x), v + 1), dtype=x.dtype)
    buf[:, 1:] = x
    outs = [ge.spec.qprob(x.to(gpu), t), ge.spec.qprob(buf.to(gpu)[:, 1:] if v > 1 else x.to(gpu), t)]
    lib = ge._lib
    h = lib.Handle(gpu.index, 1, 64)
    xd, td = x.to(gpu), torch.tensor(t, dtype=torch.float64, device=gpu)
    out = torch.full((len(x), v), -1.0, dtype=torch.float64, device=gpu)
    q = lib.QRows()
    q.size, q.kind = C.sizeof(lib.QRows), lib.Q_LOGITS_BF16 if dtype == "bf16" else lib.Q_LOGITS_F32
    q.rows, q.q, q.ld, q.temperature = len(x), xd.data_ptr(), v, td.data_ptr()
    h.call("gse_qprob", C.byref(q), v, out.data_ptr(), v, lib.stream_of(gpu.index))
    outs.append(out)
    for got in (o.cpu().numpy() for o in outs):
        assert np.isnan(got[7:]).all()
        for r in range(7):
            z = x64[r] / t[r]
            e = np.exp(z - z.max())
            np.testing.assert_allclose(got[r], e / e.sum(), rtol=1e-13, atol=1e-300)
    h.close()
