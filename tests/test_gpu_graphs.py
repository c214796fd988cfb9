"""Runs replayed from captured graphs, before and after a solver takes its long
graph, against the same runs launched kernel by kernel: equal bit for bit."""
import numpy as np
import pytest

import cases
from lbfs_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,ts", [(0, 0), (0, abi.TS_MIN), (1, 0)])
def test_graph_replays_equal_single_launches(cells, ts):
    mesh = cases.channel_mesh(20, 16, 16, seed=4)
    st = cases.smooth_state(mesh, seed=9, amp=0.004, drho=3e-4)
    x, tri = abi.rbc(4, 8.0, center=(10.0, 8.0, 8.0))
    outs = []
    for graph in (True, False):
        s = abi.Solver(mesh, abi.make_params(lattice=abi.D3Q19, visc=1.0 / 6.0, dt=0.25, body_force=(2e-5, 0.0, 0.0),
                                             time_stepping=ts, max_velocity=0.05 if ts else 0.0))
        s.set_state(*st)
        if cells:
            s.add_membranes([abi.Membrane(x, tri)])
        s.set_graph(graph)
        out = []
        # odd remainders, the last run of pairs, the run that crosses into the
        # long graph, and runs of its length with and without a rest
        for n in (5, 20, 229, 33, 64, 7):
            s.step(n)
            out += list(s.get_state())
            if cells:
                out += list(s.membrane_nodes())
        outs.append(out)
        s.close()
    for a, b in zip(*outs):
        assert np.array_equal(a, b)
