"""Transforms of small planes take X and Y in one launch with the plane in LDS:
every pair of its line lengths, few and many planes, several fields, against
numpy's transforms, relative L2 1e-13; and a pruned input, whose other lines
hold nothing."""
import pytest

import test_gpu_row_pairs as rows

pytestmark = pytest.mark.gpu

LENGTHS = [24, 32, 48, 64]


@pytest.mark.parametrize("nx", LENGTHS)
@pytest.mark.parametrize("ny", LENGTHS)
def test_lengths(gpu, nx, ny):
    for nz, nf in ((3, 1), (2, 2), (4, 3)):
        rows.test_transforms_of_nf_fields(gpu, (nx, ny, nz), nf)


@pytest.mark.parametrize("nz,nf", [(64, 1), (128, 1), (128, 2), (256, 1), (96, 3), (384, 1), (512, 1)])
@pytest.mark.parametrize("nx,ny", [(24, 64), (64, 48), (32, 32)])
def test_counts(gpu, nx, ny, nz, nf):
    rows.test_transforms_of_nf_fields(gpu, (nx, ny, nz), nf)


@pytest.mark.parametrize("shape", [(24, 64, 48), (64, 32, 24), (48, 48, 48)])
def test_pruned_gradients(gpu, shape):
    """A second LES step takes the gradients of a state known to be dealiased
    through the pruned passes: the same state as from passes that read all."""
    import os
    from ghost_amd.closure import MLP
    from ghost_amd.solvers import HDSolver
    from test_gpu_parity import grids, rel, to_gpu, to_np
    from test_gpu_small_launch import state
    got = []
    for prune in (True, False):
        g, og = grids(shape)
        s = HDSolver(g, dt=1e-3, nu=4e-3, ord=2)
        s.set_velocity([to_gpu(x) for x in state(og, 3, 501)])
        m = MLP(seed=7)
        s.set_sgs(m, 0.1)
        if not prune:
            os.environ["GHX_NO_PRUNE"] = "1"
        try:
            s.step(3)
        finally:
            os.environ.pop("GHX_NO_PRUNE", None)
        got.append([to_np(x) for x in s.velocity()])
    for a, b in zip(*got):
        assert rel(a, b) < 1e-12
