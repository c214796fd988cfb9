"""The timed kernels are those a step launches, and timed steps are whole steps."""
import numpy as np
import pytest

import cases
from lbfs_amd import abi

pytestmark = pytest.mark.gpu


# 162 nodes: membrane forces in one launch; 1442 nodes (2880 triangles): in separate passes, the
# bin scattering (mode 2) gathering the node forces itself
@pytest.mark.parametrize("freq,mode,forces", [
    (4, 0, ["mem_forces"]), (4, 1, ["mem_forces"]), (4, 2, ["mem_forces"]),
    (12, 1, ["mem_volume", "mem_edges", "mem_nodes"]), (12, 2, ["mem_volume", "mem_edges"]),
])
def test_timed_kernels_are_the_steps(freq, mode, forces):
    mesh = cases.channel_mesh(24, 16, 16, seed=14)
    x, t = abi.rbc(freq, 8.0, center=(12.0, 8.0, 8.0))
    outs = []
    for timed in (True, False):
        s = abi.Solver(mesh, abi.make_params(visc=1.0 / 6.0, dt=0.25, body_force=(2e-5, 0.0, 0.0)))
        s.set_state(*cases.smooth_state(mesh, seed=14, amp=0.005))
        s.set_ibm_binned(mode)
        s.add_membranes([abi.Membrane(x, t, **dict(abi.RBC_PARAMS, volume_ratio=0.95))])
        if timed:
            names = list(s.time_kernels(6))
            assert names == ["ibm_interp"] + forces + ["ibm_spread", "fluid", "ibm_apply"]
            assert len(s.model_bytes()) == len(names)
        else:
            s.step(6)
        outs.append(list(s.get_state()) + list(s.membrane_nodes()) + [s.membrane_globals()])
        s.close()
    for a, b in zip(*outs):
        assert np.array_equal(a, b)


def test_model_bytes_of_the_fluid_passes():
    """What each pass must move once: per cell the state in and out, inverse
    volume, force and weights (72) or gradients (48), per face its record (40)."""
    mesh = cases.channel_mesh(24, 16, 16, seed=14)
    s = abi.Solver(mesh, abi.make_params(visc=1.0 / 6.0, dt=0.25))
    n, faces = mesh.n_cells, mesh.n_faces
    assert list(s.model_bytes()) == [(16 + 72 + 4 + 12 + 16) * n + 40 * faces]
    s.set_fused(False)
    assert list(s.model_bytes()) == [(16 + 24 + 72 + 48) * n, (16 + 48 + 4 + 12 + 16) * n + 40 * faces]
    s.close()


@pytest.mark.parametrize("tile,fused", [((0, 0, 0), True), ((2, 2, 2), False), ((4, 4, 4), True), ((32, 1, 1), True)])
def test_default_fluid_pass(tile, fused):
    """Many small tiles (2304 of 2x2x2) run the two passes, others the fused one;
    either can be asked for."""
    mesh = cases.channel_mesh(32, 24, 24, seed=14)
    st = cases.smooth_state(mesh, seed=14, amp=0.005)
    s = abi.Solver(mesh, abi.make_params(visc=1.0 / 6.0, dt=0.25, tile=tile))
    names = (["gradients", "flux_update"], ["fluid"])
    assert list(s.time_kernels(1)) == names[fused]
    outs = []
    for on in (False, True):
        s.set_fused(on)
        s.set_state(*st)
        assert list(s.time_kernels(2)) == names[on]
        outs.append(np.concatenate(s.get_state()))
    s.close()
    assert np.array_equal(*outs)
