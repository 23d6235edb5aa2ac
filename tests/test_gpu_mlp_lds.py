"""The training kernel where a device gives a block less LDS than all its
waves' gradient sums take: two waves at a time, added in the same order, so the
results are the same to the bit; the network itself is made and run without
that LDS."""
import numpy as np
import pytest

from test_gpu_mlp_train import SIZES, data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", SIZES)
def test_two_waves_at_a_time(gpu, n, monkeypatch):
    import torch
    from ghost_amd.closure import MLP
    X, T = (torch.from_numpy(x).cuda() for x in data(n, 92))
    wide = MLP(91)
    monkeypatch.setenv("GHX_TRAIN_WIDE", "0")
    narrow = MLP(91)
    for a, b in zip(wide.grad(X, T), narrow.grad(X, T)):
        assert np.array_equal(np.asarray(a if isinstance(a, float) else a.cpu()),
                              np.asarray(b if isinstance(b, float) else b.cpu()))
    kw = dict(batch=n, steps=3, lr=1e-3, seed=3)
    assert np.array_equal(wide.train(X, T, **kw), narrow.train(X, T, **kw))
    assert torch.equal(wide.params(), narrow.params())
    assert torch.equal(wide.forward(X), narrow.forward(X))
