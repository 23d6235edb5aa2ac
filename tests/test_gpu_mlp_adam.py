"""Training beyond the first step: Adam (decay factors, bias correction, moments
and step count carried from step to step and from call to call) replayed in
NumPy from grad() at each step's parameters, and steps of one call against the
same steps one call each."""
import numpy as np
import pytest

from test_gpu_mlp_train import data

pytestmark = pytest.mark.gpu

B1, B2, EPS = np.float32(0.9), np.float32(0.999), np.float32(1e-8)


@pytest.mark.parametrize("n", [64, 65, 16385])
def test_steps_are_adam(gpu, n):
    """The batch is the whole set, so a step's gradient is grad()'s up to the
    order of the points: FP32 rounding of its sums, 1e-6 of the largest element.
    Elements that stay above 1e-2 of the largest agree within 1e-4 of
    themselves, and their updates (at most sqrt(steps) times the mean size of
    the gradients) within 1e-3 lr beside the parameters' own rounding."""
    import torch
    from ghost_amd.closure import MLP
    m, lr = MLP(71), np.float32(1e-2)
    X, T = (torch.from_numpy(x).cuda() for x in data(n, 72))
    m1, m2 = np.zeros(0, np.float32), np.zeros(0, np.float32)
    big = None
    for step in range(1, 6):
        p = m.params().cpu().numpy()
        loss, g = m.grad(X, T)
        g = g.cpu().numpy()
        if step == 1:
            m1, m2, big = np.zeros_like(p), np.zeros_like(p), np.ones(p.shape, bool)
        big &= np.abs(g) > 1e-2 * np.abs(g).max()
        assert big.sum() > 100
        m1 = B1 * m1 + (1 - B1) * g
        m2 = B2 * m2 + (1 - B2) * g * g
        want = p - lr * (m1 / (1 - B1 ** step)) / (np.sqrt(m2 / (1 - B2 ** step)) + EPS)
        losses = m.train(X, T, batch=n, steps=1, lr=float(lr), seed=3)
        assert abs(losses[0] - loss) <= 1e-5 * loss
        d = np.abs(m.params().cpu().numpy() - want)
        assert np.all(d[big] <= 1e-3 * lr + 2 * np.spacing(np.abs(p))[big]), (step, d[big].max())


@pytest.mark.parametrize("n", [64, 65, 16385])
def test_calls_carry_the_moments(gpu, n):
    import torch
    from ghost_amd.closure import MLP
    X, T = (torch.from_numpy(x).cuda() for x in data(n, 82))
    a, b = MLP(81), MLP(81)
    la = np.concatenate([a.train(X, T, batch=n, steps=k, lr=1e-2, seed=3) for k in (3, 2)])
    lb = np.concatenate([b.train(X, T, batch=n, steps=1, lr=1e-2, seed=3) for _ in range(5)])
    assert np.array_equal(la, lb) and torch.equal(a.params(), b.params())
