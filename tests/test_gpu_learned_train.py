"""GPU training kernels at the edges of their tiles: gradients over ragged row counts (one
row, one short of a 32-row tile, one past it, many partial sums) against the FP64 oracle,
and an epoch of Adam against the same steps in FP64."""
import numpy as np
import pytest

import mlp_oracle as mo

pytestmark = pytest.mark.gpu


def _data(n, seed):
    rng = np.random.default_rng(seed)
    X = rng.normal(size=(n, 28)).astype(np.float32)
    T = (np.tanh(X[:, :3]) * 0.5 + 0.1 * X[:, 3:6] * X[:, 25:26]).astype(np.float32)
    return X, T


def _norm(X, T):
    return [a.astype(np.float32) for a in (X.mean(0), 1 / np.maximum(X.std(0), 0.1), np.maximum(T.std(0), 0.1))]


# FP32 sums of at most 64 products per layer and `n` rows, hardware exp and reciprocal
# (1 ulp each): 2e-6 of the gradient's norm covers the six chained layers
@pytest.mark.parametrize("n", [1, 31, 32, 33, 511, 513, 4129, 20000])
def test_gradient_ragged_rows(sg, n):
    X, T = _data(n + 7, seed=n)
    mu, isig, osc = _norm(X, T)
    m = sg.MLP(seed=n)
    m.set_norm(mu, isig, osc)
    m.set_data(X, T)
    g, loss = m.gradient(n)
    Xn, Tn = mo.normalize(X[:n], T[:n], [a.astype(np.float64) for a in (mu, isig, osc)])
    lo, go = mo.loss_and_grad(m.params().astype(np.float64), Xn, Tn)
    assert abs(loss - lo) <= 2e-6 * lo
    assert np.linalg.norm(g - go) <= 2e-6 * np.linalg.norm(go)


@pytest.mark.parametrize("wg", [1, 5, 17, 40])
def test_one_batch_epoch_matches_adam(sg, wg):
    """Rows of exactly one batch: the shuffle only reorders the sums, so an epoch is one
    Adam step on the whole set; the curve holds its loss and the exported network follows."""
    n = 32 * wg
    X, T = _data(n, seed=wg)
    mu, isig, osc = _norm(X, T)
    m = sg.MLP(seed=2)
    m.set_norm(mu, isig, osc)
    m.set_data(X, T)
    w = m.params().astype(np.float64)
    Xn, Tn = mo.normalize(X, T, [a.astype(np.float64) for a in (mu, isig, osc)])
    lr, mom, var = 1e-3, np.zeros_like(w), np.zeros_like(w)
    curve = m.train(4, batch_wg=wg, lr=lr)
    for e in range(4):
        lo, g = mo.loss_and_grad(w, Xn, Tn)
        assert abs(curve[e] - lo) <= 1e-5 * lo
        mom, var = 0.9 * mom + 0.1 * g, 0.999 * var + 0.001 * g * g
        step = (0.1 * lr if e >= 3 else lr) * (mom / (1 - 0.9 ** (e + 1))) / (np.sqrt(var / (1 - 0.999 ** (e + 1))) + 1e-8)
        w = w - step
    # a gradient near zero has a relative error of up to 1 and moves its weight by up to
    # a step (1e-3) on a sign: such weights are few, so the norm holds to 1e-5
    assert np.linalg.norm(m.params() - w) <= 1e-5 * np.linalg.norm(w)
    want = mo.predict_bf16(m.params(), (X - mu) * isig) * osc
    assert np.abs(m.predict(X) - want).max() <= 2e-2 * np.abs(want).max()


def test_train_less_than_a_batch(sg):
    X, T = _data(40, seed=9)
    m = sg.MLP(seed=1)
    m.set_data(X, T)
    w = m.params()
    assert np.array_equal(m.train(3, batch_wg=2), np.zeros(3, np.float32))
    assert np.array_equal(m.params(), w)
