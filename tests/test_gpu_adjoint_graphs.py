"""Gradients whose forward run replays captured graphs between its checkpoints
against the same gradients with every step launched by itself: equal bit for
bit.  Intervals that leave the state in either buffer, and runs that cross into
the long graph."""
import numpy as np
import pytest

import cases
from lbfs_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [0, 1])
@pytest.mark.parametrize("every", [7, 8])
def test_gradients_with_graphs_equal_single_launches(cells, every):
    mesh = cases.channel_mesh(16, 12, 12, seed=4)
    st = cases.smooth_state(mesh, seed=9, amp=0.004, drho=3e-4)
    x, tri = abi.icosphere(4)
    rng = np.random.default_rng(11)
    lam_state = rng.standard_normal((mesh.n_cells, 4))
    lam_nodes = rng.standard_normal((len(x), 3)) if cells else None
    outs = []
    for graph in (True, False):
        s = abi.Solver(mesh, abi.make_params(visc=1.0 / 6.0, dt=0.25, body_force=(2e-5, 0.0, 0.0)))
        s.set_state(*st)
        if cells:
            s.add_membranes([abi.Membrane(3.5 * x + (8.0, 6.0, 6.0), tri, **abi.RBC_PARAMS)])
        s.set_graph(graph)
        out = []
        for before in (0, 193, 5):  # (the second gradient's run crosses the solver's 256th step)
            s.step(before)
            s.adjoint_forward(45, every)
            out += list(s.get_state()) + (list(s.membrane_nodes()) if cells else [])
            g = s.adjoint_backward(lam_nodes=lam_nodes, lam_state=lam_state)
            out += [g[k] for k in sorted(g)]
        s.step(9)
        out += list(s.get_state())
        outs.append(out)
        s.close()
    for a, b in zip(*outs):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)
