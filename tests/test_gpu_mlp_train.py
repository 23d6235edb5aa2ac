"""The training kernel's block partials and the fused reduction and Adam step
at the sizes where their splits change: one point, one tile, one block of four
tiles, one block more, all 256 blocks with one tile per wave, and one more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NI, NO = 10, 6
SIZES = (1, 16, 64, 65, 16384, 16385)


def data(n, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((n, NI)).astype(np.float32), rng.standard_normal((n, NO)).astype(np.float32))


@pytest.mark.parametrize("n", SIZES)
def test_gradient_matches_oracle_at_split_edges(gpu, n):
    """The oracle rounds the same operands to bfloat16; the FP32 accumulation
    order is the only difference (the bar of the network's other tests)."""
    import torch
    from ghost_amd.closure import MLP
    from oracle import oracle as O
    m = MLP(51)
    X, T = data(n, 52)
    loss, g = m.grad(torch.from_numpy(X).cuda(), torch.from_numpy(T).cuda())
    lref, gref = O.mlp_grad(m.params().cpu().numpy(), X, T, bf16=True)
    assert abs(loss - lref) < 1e-3 * lref
    g = g.cpu().numpy()
    assert np.linalg.norm(g - gref) < 2e-2 * np.linalg.norm(gref)


@pytest.mark.parametrize("n", SIZES)
def test_training_step_is_adam_on_the_gradient(gpu, n):
    """One step on the whole set against Adam's first step on grad()'s result.
    Only the order of the points differs, so an element's gradient differs by
    FP32 rounding of its sum (1e-6 of the largest): where it is above 1e-3 of
    the largest, the step lr g/(|g| + eps) agrees within 1e-3 lr."""
    import torch
    from ghost_amd.closure import MLP
    m, lr = MLP(61), 1e-3
    X, T = (torch.from_numpy(x).cuda() for x in data(n, 62))
    p0 = m.params().cpu().numpy()
    loss, g = m.grad(X, T)
    losses = m.train(X, T, batch=n, steps=1, lr=lr, seed=3)
    assert abs(losses[0] - loss) <= 1e-5 * loss
    g = g.cpu().numpy().astype(np.float64)
    big = np.abs(g) > 1e-3 * np.abs(g).max()
    assert big.any()
    d = m.params().cpu().numpy().astype(np.float64) - p0
    want = -lr * g / (np.abs(g) + 1e-8)
    ulp = np.spacing(np.abs(p0).astype(np.float32)).astype(np.float64)  # the parameters' own rounding
    assert np.all(np.abs(d - want)[big] <= 1e-3 * lr + ulp[big])
    more = m.train(X, T, batch=n, steps=3, lr=lr, seed=3)
    assert more.shape == (3,) and np.all(np.isfinite(more))
