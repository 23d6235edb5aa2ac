"""Products of 192-point rows take 12 points per lane from 4096 rows on and 6
below: one RK2 step of each solver on both sides of the line, rotating and
forced or not, against the oracle, relative L2 1e-12."""
import pytest

from test_gpu_parity import grids, rel, to_gpu, to_np
from test_gpu_small_launch import state

pytestmark = pytest.mark.gpu

SHAPES = [(192, 64, 64), (192, 48, 64), (192, 32, 128), (192, 24, 192)]


@pytest.mark.parametrize("shape", SHAPES)
def test_hd(gpu, shape):
    from ghost_amd.solvers import HDSolver
    g, og = grids(shape)
    v = state(og, 3, 301)
    s = HDSolver(g, dt=1e-3, nu=4e-3, ord=2)
    s.set_velocity([to_gpu(x) for x in v])
    og.hd_step(v, 1e-3, 4e-3, ord=2)
    s.step(1)
    for got, want in zip(s.velocity(), v):
        assert rel(to_np(got), want) < 1e-12


@pytest.mark.parametrize("shape", SHAPES)
def test_mhd(gpu, shape):
    from ghost_amd.solvers import MHDSolver
    g, og = grids(shape)
    v, a = state(og, 3, 311), state(og, 3, 312)
    s = MHDSolver(g, dt=1e-3, nu=4e-3, mu=5e-3, ord=2)
    s.set_state([to_gpu(x) for x in v], [to_gpu(x) for x in a])
    og.mhd_step(v, a, 1e-3, 4e-3, 5e-3, ord=2)
    s.step(1)
    got = s.state()
    for x, want in zip(got[0] + got[1], v + a):
        assert rel(to_np(x), want) < 1e-12


@pytest.mark.parametrize("shape", SHAPES)
def test_bouss(gpu, shape):
    from ghost_amd.solvers import BoussSolver
    g, og = grids(shape)
    v, th = state(og, 3, 321), state(og, 4, 325)[3]
    s = BoussSolver(g, dt=1e-3, nu=4e-3, kappa=5e-3, xmom=2.0, xtemp=1.5, ord=2)
    s.set_state([to_gpu(x) for x in v], to_gpu(th))
    s.set_rotation(1.5)
    og.rotbouss_step(v, th, 1e-3, 4e-3, 5e-3, 2.0, 1.5, 1.5, ord=2)
    s.step(1)
    got = s.state()
    for x, want in zip(got[0] + [got[1]], v + [th]):
        assert rel(to_np(x), want) < 1e-12
