"""Training steps of the surrogate (k_train_rows, k_train_weights) at the edges
of their blocks, against the float64 oracle (oracle/mlp_oracle.py)."""
import numpy as np
import pytest

from rapt_amd import fields as F
from rapt_amd import surrogate as S

pytestmark = pytest.mark.gpu

TENSORS = [("W1", 0, 768), ("b1", 768, 1024), ("W2", 1024, 66560), ("b2", 66560, 66816),
           ("W3", 66816, 132352), ("b3", 132352, 132608), ("W4", 132608, 133376),
           ("b4", 133376, 133379)]


@pytest.mark.parametrize("members,batch", [(1, 64), (3, 192), (4, 448), (2, 1600)])
def test_training_step_at_the_batch_edges(members, batch):
    """One Adam step on batches of one and of several 64-sample blocks, also
    not a multiple of the fragments that the weight gradients keep in flight:
    gradients of rows taken in a given order (repeats among them) against the
    float64 oracle with the same rounding points, to 1e-3 a tensor as
    the larger step's test has it; the loss;
    the new parameters against Adam on those gradients in float64 (its float32
    form rounds a handful of times: 1e-5 of the step)."""
    from oracle import mlp_oracle as O
    rng = np.random.default_rng(batch)
    th = S.init_params(batch, members)
    th[:, 768:1024] = rng.normal(0, 0.1, (members, 256))
    n = 3 * batch // 2
    X = rng.uniform(-1, 1, (n, 3)).astype(np.float32)
    T = rng.normal(0, 1, (n, 3)).astype(np.float32)
    order = rng.integers(0, n, batch)
    s = S.Surrogate(F.EarthDipole(), members=members, theta0=th)
    try:
        loss, g = s.train_steps(X, T, order, batch, 1e-3, 1e-3, want_grad=True)
        new = s.params()
    finally:
        s.close()
    for k in range(members):
        L, gr = O.loss_and_grad(th[k], X[order].astype(np.float64), T[order].astype(np.float64),
                                True)
        assert abs(loss[k] - L) <= 1e-4 * L
        for name, lo, hi in TENSORS:
            e = np.linalg.norm(g[k, lo:hi] - gr[lo:hi]) / np.linalg.norm(gr[lo:hi])
            assert e < 1e-3, (k, name, e)
        gd = g[k].astype(np.float64)
        step = 1e-3 * gd / (np.abs(gd) + 1e-8)  # the first step's m / (sqrt(v) + eps)
        assert np.max(np.abs((th[k] - new[k]) - step)) <= 1e-5 * 1e-3 + 2.0 ** -23 * np.abs(th).max()
