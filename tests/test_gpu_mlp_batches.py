"""The sensor trainer's gradient and forward at the sizes where its tiles of
32 samples and its partial sums can go wrong, against the NumPy restatement in
FP64.  Bars as in test_gpu_mlp.py: 1e-4 of each parameter block's largest
gradient entry, 1e-5 on probabilities."""
import numpy as np
import pytest

import mlp_sensor as M
from pyocfd import capi

pytestmark = pytest.mark.gpu


# one sample, the edges of a tile, a remainder, more tiles than partials
@pytest.mark.parametrize("n", [1, 31, 32, 33, 1000, 32 * 1024 + 39])
@pytest.mark.parametrize("first", [0, 5])
def test_batch_sizes_match_oracle(n, first):
    rng = np.random.default_rng(n + first)
    X = rng.standard_normal((n + first, 24)).astype(np.float32) * 0.3
    y = (rng.random(n + first) < 0.3).astype(np.float32)
    p = M.init_params(seed=3, dtype=np.float32)
    t = capi.Trainer(n + first)
    t.set_params(capi.mlp_pack(p))
    t.put(X, y)
    loss, g = t.grad(first, n, wpos=2.5)
    X64, p64 = X[first:].astype(np.float64), {k: v.astype(np.float64) for k, v in p.items()}
    loss_ref, g_ref = M.loss_and_grads(p64, X64, y[first:].astype(np.float64), wpos=2.5)
    assert abs(loss - loss_ref) <= 1e-5 * abs(loss_ref)
    gg = capi.mlp_unpack(g)
    for k in g_ref:
        err = np.abs(gg[k] - g_ref[k]).max() / max(np.abs(g_ref[k]).max(), 1e-30)
        assert err <= 1e-4, (k, err)
    prob_ref, _ = M.forward(p64, X64)
    assert np.abs(t.predict(first, n) - prob_ref).max() <= 1e-5


@pytest.mark.parametrize("n", [1, 17, 33])
def test_lanes_past_the_last_sample_add_nothing(n):
    """A bias that the samples' own inputs cancel: their activations are
    ordinary, those of a zero input overflow the derivative of the GELU.  Bar as
    above."""
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, 24)).astype(np.float32) * 0.3
    X[:, 0] = 1.0
    y = (rng.random(n) < 0.5).astype(np.float32)
    p = M.init_params(seed=3, dtype=np.float32)
    p["W1"][0] = 0.0
    p["W1"][0, 0], p["b1"][0] = -1e25, 1e25
    t = capi.Trainer(n)
    t.set_params(capi.mlp_pack(p))
    t.put(X, y)
    loss, g = t.grad(0, n, wpos=2.5)
    loss_ref, g_ref = M.loss_and_grads({k: v.astype(np.float64) for k, v in p.items()}, X.astype(np.float64),
                                       y.astype(np.float64), wpos=2.5)
    assert abs(loss - loss_ref) <= 1e-5 * abs(loss_ref)
    gg = capi.mlp_unpack(g)
    for k in g_ref:
        assert np.abs(gg[k] - g_ref[k]).max() <= 1e-4 * np.abs(g_ref[k]).max(), k
