"""Lines of 3 * 2^k points (24 .. 384) in radix-6, 8 and 4 stages, along each
axis and next to axes that fill neither a wavefront nor a tile: one RK2 step of
each solver with the tracers' velocities and the extrema, against the oracle,
relative L2 1e-12 (the transforms of one to three fields alone are in
test_gpu_row_pairs)."""
import numpy as np
import pytest

from test_gpu_parity import grids, rel, to_gpu, to_np
from test_gpu_small_launch import state

pytestmark = pytest.mark.gpu

LENGTHS = [24, 48, 96, 192, 384]
SHAPES = [(n, 24, 16) for n in LENGTHS] + [(24, n, 16) for n in LENGTHS] + [(16, 24, n) for n in LENGTHS] + [
    (192, 48, 64), (96, 96, 48), (48, 192, 96), (24, 64, 384)]


@pytest.mark.parametrize("shape", SHAPES)
def test_hd(gpu, shape):
    from ghost_amd.lagpart import GPart
    from ghost_amd.solvers import HDSolver
    g, og = grids(shape)
    v = state(og, 3, 301)
    s = HDSolver(g, dt=1e-3, nu=4e-3, ord=1)
    s.set_velocity([to_gpu(x) for x in v])
    p = GPart(g, 40)
    rng = np.random.default_rng(302)
    pos = [rng.uniform(0.0, n, 40) for n in shape]
    p.set_positions(*[to_gpu(x) for x in pos])
    s.set_tracers(p)
    og.hd_step(v, 1e-3, 4e-3, ord=1)
    s.step(1)
    for got, want in zip(s.velocity(), v):
        assert rel(to_np(got), want) < 1e-12
    ref = [x.copy() for x in pos]
    og.tracer_stage(v, ref, [x.copy() for x in pos], 1e-3, 1.0, ghost_solve=False)
    for x, want, n in zip(p.positions(), ref, shape):
        d = np.mod(to_np(x) - want + n / 2, n) - n / 2
        assert np.max(np.abs(d)) < 1e-10
    V = [to_gpu(x) for x in v]
    for kin in (0, 1):
        assert g.maxabs(*V, kin) == pytest.approx(og.maxabs(*v, kin), rel=1e-12)


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
