"""Members read and written between replays of the captured step: the graph is
kept, the states are checked again, and one that holds modes outside the
dealias set takes the eager step.  The same kernels run on the same values as
without a graph, so the states agree bit for bit."""
import numpy as np
import pytest
import torch

from test_gpu_small_launch import state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(16,), (16, 24, 24, 32)])
def test_reads_and_writes_between_steps(gpu, sizes):
    from ghost_amd.solvers import Ensemble
    from test_gpu_parity import grids, to_gpu
    start = [[to_gpu(x) for x in state(grids((n, n, n))[1], 3, 401 + m)] for m, n in enumerate(sizes)]
    both = []
    for graph in (True, False):
        e = Ensemble(list(sizes), [4e-3 + 1e-3 * m for m in range(len(sizes))], dt=1e-3, ord=2)
        e.set_graph(graph)
        seen = []
        for m, v in enumerate(start):
            e.set_velocity(m, v)
        for turn in range(4):
            e.step(2)
            e.sync()
            seen.append([x.clone() for m in range(len(sizes)) for x in e.velocity(m)])
            if turn == 1:  # a mode outside the dealias set in the last member
                m, n = len(sizes) - 1, sizes[-1]
                v = e.velocity(m)
                v[1][n // 2 - 1, 2, 3] = 0.25 - 0.5j
                e.set_velocity(m, v)
        both.append(seen)
    for a, b in zip(*both):
        for x, y in zip(a, b):
            assert torch.equal(x, y)
    assert not np.any([torch.equal(x, y) for x, y in zip(both[0][0], both[0][3])])
