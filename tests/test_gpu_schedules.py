"""The step schedules on a mesh beyond those that run on one stream, with a
membrane whose forces take separate passes and with one whose forces take one
launch: equal bit for bit."""
import numpy as np
import pytest

import cases
from lbfs_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("freqs", [(12, 4), (4, 3)])
@pytest.mark.parametrize("mode", [1, 2])
def test_schedules_of_two_streams_are_bitwise_equal(freqs, mode):
    mesh = cases.channel_mesh(64, 48, 48, seed=14)
    assert mesh.n_cells > 128 * 1024
    st = cases.smooth_state(mesh, seed=14, amp=0.005)
    mems = [abi.Membrane(*abi.rbc(f, 14.0, center=(16.0 + 32.0 * k, 24.0, 24.0)),
                         **dict(abi.RBC_PARAMS, volume_ratio=0.95)) for k, f in enumerate(freqs)]
    outs = []
    for schedule in (0, 1, 2):
        for graph in (True, False):
            s = abi.Solver(mesh, abi.make_params(visc=1.0 / 6.0, dt=0.25, body_force=(2e-5, 0.0, 0.0)))
            s.set_state(*st)
            s.set_step_schedule(schedule)
            s.set_graph(graph)
            s.set_ibm_binned(mode)
            s.add_membranes(mems)
            s.step(8)
            outs.append(list(s.get_state()) + list(s.membrane_nodes()) + [s.cell_force(), s.membrane_globals()])
            s.close()
    for o in outs[1:]:
        for a, b in zip(outs[0], o):
            assert np.array_equal(a, b)
