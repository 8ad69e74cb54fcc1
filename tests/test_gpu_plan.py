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
