"""An ensemble with more members than their fields fit a launch grid's y or z
extent (65535): 22000 members of 8^3, whose y inverses would split into 132000
blocks and whose states are 66000 fields to look at.  Members around the limits
against the same runs alone; the last one holds modes outside the dealias set,
so the look at the states has to reach it."""
import numpy as np
import pytest

from test_gpu_parity import grids, rel, to_gpu, to_np
from test_gpu_small_launch import state

pytestmark = pytest.mark.gpu

N, COUNT = 8, 22000
MEMBERS = [0, 1, 10921, 10922, 10923, 21844, 21845, COUNT - 1]


def test_members_beyond_a_grid_extent(gpu):
    from ghost_amd.solvers import Ensemble
    og = grids((N, N, N))[1]
    e = Ensemble([N] * COUNT, [4e-3] * COUNT, dt=1e-3, ord=2)
    start = {}
    for m in MEMBERS:
        start[m] = [to_gpu(x) for x in state(og, 3, 501 + m)]
    start[COUNT - 1][1][3, 2, 3] = 0.25 - 0.5j
    want = {}
    for m, v in start.items():
        e.set_velocity(m, v)
        one = Ensemble([N], [4e-3], dt=1e-3, ord=2)
        one.set_velocity(0, v)
        one.step(2)
        want[m] = [to_np(x) for x in one.velocity(0)]
    e.step(2)
    for m in MEMBERS:
        for x, y in zip(e.velocity(m), want[m]):
            assert rel(to_np(x), y) < 1e-13, m
    assert all(not np.any(to_np(x)) for x in e.velocity(2))
