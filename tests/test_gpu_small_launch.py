"""Both sides of the lines at which the substeps change kernels: one field per
block and one lane group per component below 3328 kept lines (kx, ky) or
(kx, z), every field in turn above, and the y inverse by field again from
10000.  nx = 384 keeps 129 kx, so 24 lines along an axis are below (3096), 32
above (4128) and 96 far above (12384).  One RK2 step of each solver against the
oracle, relative L2 1e-12."""
import numpy as np
import pytest

from test_gpu_parity import grids, rel, to_gpu, to_np

pytestmark = pytest.mark.gpu

# z lines of 8 and 6 points per lane, of 512 points, and of one lane
SHAPES = [(384, 24, 64), (384, 32, 64), (384, 32, 24), (384, 32, 4), (384, 64, 32), (384, 16, 96), (384, 32, 512),
          (384, 24, 48)]


def state(og, n, seed):
    """Dealiased fields of unit size: the library's own solenoidal initial
    fields where components are asked in threes, one more for a scalar."""
    out = []
    while len(out) < n:
        out += og.initialv_k4exp(3.0, 1.0, seed + len(out))[0]
    return out[:n]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("rotating", [False, True])
def test_hd(gpu, shape, rotating):
    from ghost_amd.solvers import HDSolver
    g, og = grids(shape)
    v, f = state(og, 3, 201), og.initialfv_random(2.0, 3.0, 0.3, 202)[0]
    s = HDSolver(g, dt=1e-3, nu=4e-3, ord=2)
    s.set_velocity([to_gpu(x) for x in v])
    s.set_forcing([to_gpu(x) for x in f])
    if rotating:
        s.set_rotation(2.5)
        og.roth_step(v, 1e-3, 4e-3, 2.5, f=f, ord=2)
    else:
        og.hd_step(v, 1e-3, 4e-3, f=f, ord=2)
    s.step(1)
    for got, want in zip(s.velocity(), v):
        assert rel(to_np(got), want) < 1e-12


@pytest.mark.parametrize("shape", SHAPES)
def test_mhd(gpu, shape):
    from ghost_amd.solvers import MHDSolver
    g, og = grids(shape)
    v, a = state(og, 3, 211), state(og, 3, 212)
    f, m = og.initialfv_random(2.0, 3.0, 0.3, 213)[0], og.initialfv_random(1.0, 2.0, 0.2, 214)[0]
    s = MHDSolver(g, dt=1e-3, nu=4e-3, mu=5e-3, ord=2)
    s.set_state([to_gpu(x) for x in v], [to_gpu(x) for x in a])
    s.set_forcing([to_gpu(x) for x in f], [to_gpu(x) for x in m])
    og.mhd_step(v, a, 1e-3, 4e-3, 5e-3, f=f, m=m, ord=2)
    s.step(1)
    got = s.state()
    for x, want in zip(got[0] + got[1], v + a):
        assert rel(to_np(x), want) < 1e-12


@pytest.mark.parametrize("shape", SHAPES)
def test_bouss_with_tracers(gpu, shape):
    """Order 1 updates the fields in place over the state the nonlinear terms
    read; tracers take the spline z inverse."""
    from ghost_amd.lagpart import GPart
    from ghost_amd.solvers import BoussSolver
    for ord_ in (1, 2):
        g, og = grids(shape)
        v, th = state(og, 3, 221), state(og, 4, 225)[3]
        th[0, 0, 0] = 2.0
        s = BoussSolver(g, dt=1e-3, nu=4e-3, kappa=5e-3, xmom=2.0, xtemp=1.5, ord=ord_)
        s.set_state([to_gpu(x) for x in v], to_gpu(th))
        s.set_forcing(None, None)
        s.set_rotation(1.5)
        p = GPart(g, 50)
        rng = np.random.default_rng(226)
        pos = [rng.uniform(0.0, n, 50) for n in shape]
        p.set_positions(*[to_gpu(x) for x in pos])
        s.set_tracers(p)
        og.rotbouss_step(v, th, 1e-3, 4e-3, 5e-3, 2.0, 1.5, 1.5, ord=ord_)
        s.step(1)
        got = s.state()
        for x, want in zip(got[0] + [got[1]], v + [th]):
            assert rel(to_np(x), want) < 1e-12
        if ord_ == 1:  # one stage on the new velocity (the exact spline solve: GHOST's slips on short axes)
            ref = [x.copy() for x in pos]
            og.tracer_stage(v, ref, [x.copy() for x in pos], 1e-3, 1.0, ghost_solve=False)
            for x, want, n in zip(p.positions(), ref, shape):
                d = np.mod(to_np(x) - want + n / 2, n) - n / 2
                assert np.max(np.abs(d)) < 1e-10
