"""The network's fused passes at the edges of their tiles (16 samples a tile, 256 a turn of the weight
gradients, 1024 blocks of the forward pass) against the FP64 oracle."""
import numpy as np
import pytest

import mlp_oracle as MO


def _set(n, seed):
    rng = np.random.default_rng(seed)
    X = np.zeros((n, 6), np.float32)
    X[:, 0] = rng.uniform(-1, 2, n)
    X[:, 1] = rng.uniform(0, 1.5, n)
    X[:, 2] = rng.uniform(-1, 1, n)
    X[np.arange(n), 3 + rng.integers(0, 3, n)] = 1
    y = rng.integers(0, 8, n).astype(np.int32)
    return X, y


def _params(seed):
    p = MO.init_params(seed)
    return (p + 0.05 * np.random.default_rng(seed).standard_normal(p.size)).astype(np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 15, 16, 17, 255, 257, 1023, 1025, 16385])
def test_gpu_mlp_tiles(ctx, n):
    X, y = _set(n, n)
    p = _params(5)
    Lo, go = MO.loss_grad(p.astype(np.float64), X, y)
    L, g = ctx.mlp_loss_grad(X, y, p)
    # FP32 sums of at most 70 products per layer, four layers each way: 1e-5 of the norm
    assert abs(L - Lo) <= 1e-5 * abs(Lo)
    assert np.linalg.norm(g - go) <= 1e-5 * np.linalg.norm(go)
    Z, _ = MO.forward(p.astype(np.float64), X)
    assert np.abs(ctx.mlp_infer(X, p) - MO.softmax(Z)).max() < 2e-5


@pytest.mark.gpu
@pytest.mark.parametrize("n,batch", [(1, 1), (33, 33), (300, 1000), (1000, 272)])
def test_gpu_mlp_first_steps(ctx, n, batch):
    """One epoch: the loss is that of the first minibatch; with a single minibatch every parameter with a
    gradient moves by lr against its sign (Adam's first step)."""
    X, y = _set(n, n)
    p0 = _params(6)
    lr = 1e-3
    p, losses = ctx.mlp_train(X, y, p0, epochs=1, batch=batch, lr=lr, seed=2)
    assert len(losses) == 1 and np.isfinite(losses[0]) and np.isfinite(p).all()
    if batch >= n:
        Lo, go = MO.loss_grad(p0.astype(np.float64), X, y)
        assert abs(losses[0] - Lo) <= 1e-5 * abs(Lo)
        step = p.astype(np.float64) - p0
        # eps = 1e-8 against |g| and an FP32 rounding of p (|p| < 4: 2.4e-7)
        big = np.abs(go) > 1e-3 * np.abs(go).max()
        assert np.abs(step[big] + lr * np.sign(go[big])).max() < 1e-2 * lr
        assert np.abs(step).max() <= lr * 1.001 + 2.4e-7
