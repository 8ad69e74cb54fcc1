"""GPU parity of the split-row finish's plan, on the split-row path (no row of these may need the exact path): rows whose
min-p cut lies far before their top-p cut, rows that keep everything, rows whose logits range far past the fine
histogram bins."""
import numpy as np
import pytest
import torch

from oracle import sampling_ref as ora

pytestmark = pytest.mark.gpu


def _zipf(rng, n, v):
    """Normals on a Zipf slope over a random ranking: the maximum is 25 or more above most tokens."""
    x = rng.normal(0.0, 2.5, size=(n, v)) - 1.1 * np.log1p(rng.permuted(np.tile(np.arange(v), (n, 1)), axis=1))
    return x.astype(np.float32)


def _check(ge, gpu, x, params, seed):
    n, v = x.shape
    u = np.array([ora.uniform(seed + r, 5) for r in range(n)], np.float64)
    sel = ge.sampling.sample_ex(torch.from_numpy(x).to(gpu), params, None, None, None, uniforms=u)
    paths = ge._lib.handle(gpu.index, n, v).row_paths(n)
    assert sel.tolist() == ora.sample(x, params, None, None, None, uniforms=u)
    assert (paths == ge._lib.PATH_EXACT).sum() == 0, paths
    return paths


@pytest.mark.parametrize("v", [29001, 151936])
def test_min_p_before_top_p(ge, gpu, v):
    """Flat rows (thousands of elements between the min-p and the top-p cut, either one first), min-p at, just above and
    just below a bin edge of the histogram."""
    rng = np.random.default_rng(v)
    P = ge.sampling.SamplingParams
    mps = [0.05, 0.02, 0.3, float(np.exp(-3.0)), float(np.exp(-3.0) * (1 + 1e-7)), float(np.exp(-3.0) * (1 - 1e-7)),
           1e-6, 1e-12]
    params = [P(temperature=1.2 + 0.1 * (r % 4), top_p=[0.999, 0.9, 1.0][r % 3], min_p=mps[r % 8]) for r in range(24)]
    x = rng.normal(0.0, 1.5, size=(24, v)).astype(np.float32)
    paths = _check(ge, gpu, x, params, 77)
    assert (paths == ge._lib.PATH_DEEP).sum() > 0


@pytest.mark.parametrize("v", [50257, 128256])
def test_keep_all_and_long_tails(ge, gpu, v):
    """top_p 1 and top_p just below it, from low to high temperatures, over rows whose tail holds most of the
    vocabulary."""
    rng = np.random.default_rng(v)
    P = ge.sampling.SamplingParams
    params = [P(temperature=[0.3, 0.7, 1.0, 1.4][r % 4], top_p=[1.0, 1.0, 0.9999, 1.0 - 1e-7][r // 4 % 4])
              for r in range(32)]
    _check(ge, gpu, _zipf(rng, 32, v), params, 991)
    flat = rng.normal(0.0, 1.0, size=(8, v)).astype(np.float32)
    paths = _check(ge, gpu, flat, [P(temperature=1.0) for _ in range(8)], 17)
    assert (paths == ge._lib.PATH_DEEP).sum() > 0


@pytest.mark.parametrize("n,v,dtype", [(512, 262144, "bf16"), (256, 151936, "f32")])
def test_cuts_far_below_the_maximum(ge, gpu, n, v, dtype):
    """Large batches of wide flat rows whose top-p cut lies 12 to 16 below the maximum (slices of 64K tokens: what one
    slice lists of a window must fit its LDS list): all of them on the split-row pass, tokens of every 32nd row against
    the oracle."""
    g = torch.Generator(device=gpu).manual_seed(v)
    x = torch.randn((n, v), generator=g, device=gpu).mul_(2.5)
    x = x.bfloat16() if dtype == "bf16" else x
    P = ge.sampling.SamplingParams
    params = [P(temperature=1.0, top_p=[0.998, 0.999, 0.9995][r % 3]) for r in range(n)]
    u = np.random.default_rng(v).random(n)
    sel = ge.sampling.sample_ex(x, params, None, None, None, uniforms=u)
    paths = ge._lib.handle(gpu.index, n, v).row_paths(n)
    assert (paths == ge._lib.PATH_EXACT).sum() == 0, (paths == ge._lib.PATH_EXACT).sum()
    assert (paths == ge._lib.PATH_DEEP).sum() > n // 2
    some = list(range(0, n, 32))
    want = ora.sample(x[some].float().cpu().numpy(), [params[r] for r in some], None, None, None, uniforms=u[some])
    assert [sel.tolist()[r] for r in some] == want


def test_dist_of_long_tails(ge, gpu):
    """dist over such rows: every probability against the oracle's."""
    rng = np.random.default_rng(4)
    n, v = 8, 50257
    P = ge.sampling.SamplingParams
    params = [P(temperature=[0.8, 1.0][r % 2], top_p=[1.0, 0.9999][r // 2 % 2], min_p=[0.0, 1e-7][r // 4]) for r in range(n)]
    x = _zipf(rng, n, v)
    d = ge.sampling.dist_batch(torch.from_numpy(x).to(gpu), params).cpu().numpy()
    paths = ge._lib.handle(gpu.index, n, v).row_paths(n)
    assert (paths == ge._lib.PATH_EXACT).sum() == 0, paths
    for r in range(n):
        np.testing.assert_allclose(d[r], ora.dist(x[r], params[r]), rtol=1e-12, atol=1e-300)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_draws_settled_in_the_head(ge, gpu, dtype):
    """Rows whose keep set runs past the certified head but whose draw mostly falls inside it: small batches over one
    long vocabulary (many parts a row) and larger ones, every cut alone and together, uniforms from 0 to just below 1.
    Tokens against the oracle on both paths; most rows end in the main pass."""
    v = 100003
    rng = np.random.default_rng(31)
    P = ge.sampling.SamplingParams
    cuts = [dict(top_p=0.9), dict(top_p=0.97), dict(), dict(top_k=3000, top_p=0.999), dict(min_p=1e-4),
            dict(top_k=400, top_p=0.95, min_p=1e-3)]
    us = [0.0, 2.0 ** -53, 0.1, 0.5, 0.75, 0.9, 0.97, 1.0 - 2.0 ** -53]
    for n in (1, 6, 48):
        main = 0
        for rep in range(8 if n == 1 else 1):
            x = torch.from_numpy(_zipf(rng, n, v))
            x = x.bfloat16() if dtype == "bf16" else x
            params = [P(temperature=[0.7, 1.0, 1.3][(r + rep) % 3], **cuts[(r + rep) % 6]) for r in range(n)]
            u = np.array([us[(r // 2 + rep) % 8] for r in range(n)])
            sel = ge.sampling.sample_ex(x.to(gpu), params, None, None, None, uniforms=u)
            paths = ge._lib.handle(gpu.index, n, v).row_paths(n)
            assert sel.tolist() == ora.sample(x.float().numpy(), params, None, None, None, uniforms=u), (n, rep)
            main += int((paths == ge._lib.PATH_MAIN).sum())
        assert main >= (4 if n == 1 else n // 2), (n, main)


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("n,v,order", [(n, v, o) for n, v in [(1, 128256), (4, 131072), (2, 262144), (8, 32000), (1, 9000)]
                                       for o in ("falling", "none")] + [(4, 131072, "one part")])
def test_best_tokens_in_one_part(ge, gpu, n, v, dtype, order):
    """Rows whose ids are ordered by rank, or whose best tokens fill one part of the main pass: greedy and nucleus rows
    with 20 and 64 logprobs and top-k rows need no exact path, and the ordered top-k rows end in the main pass (a part in
    any order lists within a fifth of its target, 48 here: some rows fall short of their 40)."""
    rng = np.random.default_rng(v + n)
    x = _zipf(rng, n, v)
    x -= x.mean(axis=1, keepdims=True)  # (ordered parts span little: near 0 their values stay apart in 16 key bits)
    if order != "none":
        x = -np.sort(-x, axis=1)
    if order == "one part":  # (part 8 of 16, in any order)
        x = np.concatenate([rng.permuted(x[:, 8192:v // 2 + 8192], axis=1), rng.permuted(x[:, :8192], axis=1),
                            x[:, v // 2 + 8192:]], axis=1)
    x = torch.from_numpy(x)
    x = x.bfloat16() if dtype == "bf16" else x
    x32, xd = x.float().numpy(), x.to(gpu)
    P = ge.sampling.SamplingParams
    u = rng.random(n)
    for p in (P(logprobs=20), P(logprobs=64), P(temperature=0.9, top_p=0.9, logprobs=20),
              P(temperature=0.9, top_p=0.9, logprobs=64), P(temperature=0.8, top_k=40, top_p=0.95),
              P(temperature=0.8, top_k=40)):
        sel = ge.sampling.sample_ex(xd, [p] * n, None, None, None, uniforms=u)
        paths = ge._lib.handle(gpu.index, n, v).row_paths(n)
        want = ora.sample_full(x32, [p] * n, None, None, None, None, u)
        assert sel.tolist() == [w["token"] for w in want], p
        assert (paths == ge._lib.PATH_EXACT).sum() == 0, (p, paths)
        if p.top_k and order != "one part":
            assert (paths == ge._lib.PATH_MAIN).all(), (p, paths)
        if p.logprobs:
            ids = sel.logprob_ids.cpu().numpy()
            for r in range(n):
                assert list(ids[r, :p.logprobs]) == list(want[r]["logprob_ids"]), p


@pytest.mark.parametrize("parts", [6, 16])
def test_bound_past_the_sum(ge, gpu, parts):
    """Logits of 2^27 (a ulp apart: 8) make the bound on the unlisted mass (1.8e-7 |z| relative) larger than the whole
    sum: the head cannot even tell that its first rank is kept, and the split-row pass decides."""
    v = parts * 8192
    x = np.full((4, v), 2.0 ** 27 - 8, np.float32)
    for p in range(parts):  # (40 lanes of every part's sample hold a maximum: the parts list these and no more)
        x[:, p * 8192:p * 8192 + 2048:50] = 2.0 ** 27
    P = ge.sampling.SamplingParams
    paths = _check(ge, gpu, x, [P(temperature=1.0, top_p=[0.5, 0.8, 0.3, 0.7][r]) for r in range(4)], 5)
    assert (paths == ge._lib.PATH_DEEP).any()


def test_masked_rows_whose_samples_are_empty(ge, gpu):
    """Masked rows whose allowed runs lie outside most parts' samples (those parts start listing everything). Greedy rows
    with logprobs, sampled rows with and without, T = 1 and not: tokens, ids and logprobs against the oracle, none on the
    exact path."""
    v, n = 151936, 12
    rng = np.random.default_rng(8)
    x = rng.normal(0.0, 2.0, size=(n, v)).astype(np.float32)
    masks = np.zeros((n, v), bool)
    for r in range(n):
        for s in range(18):  # (runs of 400 tokens past the first 2048 of every 8192)
            masks[r, s * 8192 + 4000 + 7 * r:s * 8192 + 4400 + 7 * r] = True
    P = ge.sampling.SamplingParams
    params = [[P(logprobs=7), P(temperature=1.0, top_p=0.9, logprobs=20), P(temperature=0.8, top_k=50)][r % 3]
              for r in range(n)]
    u = rng.random(n)
    sel = ge.sampling.sample_ex(torch.from_numpy(x).to(gpu), params, None, None, [torch.from_numpy(m) for m in masks],
                                uniforms=u)
    paths = ge._lib.handle(gpu.index, n, v).row_paths(n)
    want = ora.sample_full(x, params, None, None, list(masks), None, u)
    assert sel.tolist() == [w["token"] for w in want]
    ids, lps = sel.logprob_ids.cpu().numpy(), sel.logprobs.cpu().numpy()
    for r in range(n):
        if params[r].logprobs:
            k = params[r].logprobs
            assert list(ids[r, :k]) == list(want[r]["logprob_ids"])
            np.testing.assert_allclose(lps[r, :k], want[r]["logprobs"], rtol=2e-7)
    assert (paths == ge._lib.PATH_EXACT).sum() == 0, paths


@pytest.mark.parametrize("flags", [0, 16])
@pytest.mark.parametrize("v", [9001, 50257, 151936])
def test_window_lists_of_ties(ge, gpu, v, flags):
    """Flat rows with tie groups of tens to thousands of elements at the cut and at the draw (bf16 logits; fp32 logits on
    a grid), so that the window lists are long and their key buckets crowded: tokens against the oracle, by the sorted
    finish and by the sub-bin walk (GSE_BATCH_SUBBIN_FINISH)."""
    assert ge._lib.BATCH_SUBBIN_FINISH == 16
    n = 16
    rng = np.random.default_rng(v)
    P = ge.sampling.SamplingParams
    params = [P(temperature=[1.0, 0.7, 1.6, 1.0][r % 4], top_p=[0.95, 0.8, 1.0, 0.999][r // 4], min_p=[0.0, 0.03][r % 2])
              for r in range(n)]
    base = rng.normal(0.0, 2.0, size=(n, v)).astype(np.float32)
    u = np.array([ora.uniform(r, 11) for r in range(n)], np.float64)
    for x in (torch.from_numpy(base).bfloat16(), torch.from_numpy(np.round(base * 16) / 16),
              torch.from_numpy(np.round(base * 64) / 64)):
        sel = ge.sampling.sample_ex(x.to(gpu), params, None, None, None, uniforms=u, flags=flags)
        paths = ge._lib.handle(gpu.index, n, v).row_paths(n)
        assert sel.tolist() == ora.sample(x.float().numpy(), params, None, None, None, uniforms=u)
        # (a finish that fails its checks hands its row to the exact path, which would hide it)
        assert (paths == ge._lib.PATH_DEEP).any() and not (paths == ge._lib.PATH_EXACT).any(), paths


@pytest.mark.parametrize("step", [64, 16])
def test_tie_groups_around_the_counting_limit(ge, gpu, step):
    """Rows of tie groups of one size each, from a few members to more than the finish ranks by counting, with one to four
    groups in a window (grid steps of 1/64 and 1/16 against bins of 1/32)."""
    sizes = [48, 64, 65, 128, 193, 255, 256, 257, 341, 342, 511, 512, 513, 700, 1024, 1025]
    n, v = len(sizes), 40000
    rng = np.random.default_rng(step)
    P = ge.sampling.SamplingParams
    x = np.empty((n, v), np.float32)
    for r, g in enumerate(sizes):
        x[r] = 4.0 - (rng.permutation(v) // g).astype(np.float32) / step
    for top_p in (0.9, 1.0):
        params = [P(temperature=1.0, top_p=top_p) for _ in range(n)]
        u = np.array([ora.uniform(r, 3) for r in range(n)], np.float64)
        sel = ge.sampling.sample_ex(torch.from_numpy(x).to(gpu), params, None, None, None, uniforms=u)
        paths = ge._lib.handle(gpu.index, n, v).row_paths(n)
        assert sel.tolist() == ora.sample(x, params, None, None, None, uniforms=u)
        assert (paths == ge._lib.PATH_DEEP).any() and not (paths == ge._lib.PATH_EXACT).any(), paths
