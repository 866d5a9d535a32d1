"""Training gradients where a gradient step's blocks and passes end: fewer
rows than a block's 32, its edges, and more rows than one pass of all blocks;
inference where a wave's 16-row tiles end."""

import numpy as np
import pytest

from oracle.mlp_ref import forward_backward, infer_bf16
from scs_amd import scs

pytestmark = pytest.mark.gpu


def _model(seed):
    d = scs.model_init(seed).to_arrays()
    d["mean"][:6] = [10, 100, 3, 30, 15, 2]
    d["scale"][:6] = [0.17, 0.017, 0.7, 0.06, 0.12, 0.9]
    rng = np.random.default_rng(seed)
    d["b1"], d["b2"] = (rng.normal(0, 0.1, 64).astype(np.float32) for _ in range(2))
    return scs.Model.from_arrays(d), d


def _rows(n):
    rng = np.random.default_rng(n)
    X = np.stack([rng.integers(0, 20, n), rng.integers(0, 200, n), rng.integers(1, 6, n),
                  rng.integers(1, 60, n), rng.integers(1, 30, n), rng.random(n) * 4],
                 axis=1).astype(np.float32)
    return X, (rng.random(n) < 0.3).astype(np.float32)


@pytest.mark.parametrize("n", [1, 31, 32, 33, 2049, 8192, 8225])
def test_gradient_of_odd_batches(n):
    m, d = _model(3)
    X, y = _rows(n)
    g, loss = scs.mlp_grad(m, X, y, pos_weight=2.5)
    rl, rg = forward_backward(d, X, y, pos_weight=2.5)
    got = g.to_arrays()
    # a value passes through at most about 200 FP32 roundings (64 + 64 products
    # of the two layers and the sums over 32 rows and the blocks), each of at
    # most 6e-8 of the largest term: 1.2e-5 of the largest gradient, and 1e-4
    # leaves room for terms that cancel
    for k in ("w1", "b1", "w2", "b2", "w3", "b3"):
        ref = np.asarray(rg[k])
        have = got[k][:6] if k == "w1" else got[k]
        ref = ref[:6] if k == "w1" else ref
        assert np.abs(have - ref).max() <= 1e-4 * max(np.abs(ref).max(), 1e-3), (k, n)
    assert abs(loss - rl) <= 1e-4 * max(1.0, abs(rl))


@pytest.mark.parametrize("n", [1, 15, 16, 17, 65537])
def test_inference_of_odd_row_counts(n):
    m, d = _model(5)
    X, _ = _rows(n)
    ref = infer_bf16(d, X)
    # the bounds of the BF16 comparison on 1,000 rows
    assert np.allclose(scs.mlp_infer(m, X), ref, rtol=2e-2,
                       atol=2e-2 * max(1.0, float(np.abs(ref).max())))
