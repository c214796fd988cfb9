"""Membranes whose coordinates lie beyond the integers of the grid's indices, as
those of a run that has blown up: their stencils stay off the grid (between
walls) or wrap onto it, and never leave its arrays."""
import numpy as np
import pytest

import cases
from lbfs_amd import abi

pytestmark = pytest.mark.gpu


def solver(periodic, axis=None, far=None, kernel=abi.IBM_COS4, mode=-1):
    mesh = abi.HexMesh(20, 18, 16, periodic=periodic, jitter=0.1, seed=3)
    s = abi.Solver(mesh, abi.make_params(visc=1.0 / 6.0, dt=0.25, body_force=(2e-5, 0.0, 0.0)))
    s.set_state(*cases.smooth_state(mesh, seed=3, amp=0.005))
    if axis is not None:
        s.set_ibm_binned(mode)
        x, t = abi.rbc(4, 8.0, center=(10.0, 9.0, 8.0))
        if far is not None:
            x[:, axis] = far + 1e-4 * far * x[:, axis]  # (stretched: its nodes stay apart in single precision)
        s.add_membranes([abi.Membrane(x, t, **abi.RBC_PARAMS)], ibm_kernel=kernel)
    return s


@pytest.mark.parametrize("kernel", [abi.IBM_COS4, abi.IBM_LINEAR2, abi.IBM_LAGRANGE4])
@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_nodes_beyond_the_grid(kernel, mode, axis):
    walled = solver((0, 0, 0))
    walled.step(4)
    want = walled.get_state()
    walled.close()
    for far in (3e9, -3e9, 1e15, -1e15):
        print("axis %d, kernel %d, mode %d, at %g" % (axis, kernel, mode, far), flush=True)
        s = solver((0, 0, 0), axis, far, kernel, mode)
        s.step(4)
        got = s.get_state()
        s.close()
        if kernel != abi.IBM_LAGRANGE4:  # (which takes the planes nearest to a node, however far)
            for a, b in zip(want, got):
                assert np.array_equal(a, b)
        s = solver((1, 1, 1), axis, far, kernel, mode)
        s.step(4)
        s.get_state()
        s.close()


@pytest.mark.parametrize("axis", [0, 1, 2])
def test_gradient_with_nodes_beyond_the_grid(axis):
    for far in (3e9, -1e15):
        print("axis %d at %g" % (axis, far), flush=True)
        s = solver((0, 0, 0), axis, far)
        s.adjoint_forward(5, 2)
        rng = np.random.default_rng(1)
        g = s.adjoint_backward(lam_state=rng.standard_normal((s.n, 4)))
        s.close()
        p = solver((0, 0, 0))
        p.adjoint_forward(5, 2)
        rng = np.random.default_rng(1)
        h = p.adjoint_backward(lam_state=rng.standard_normal((p.n, 4)))
        p.close()
        assert np.array_equal(g["state0"], h["state0"])


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("periodic", [(0, 0, 0), (1, 1, 1)])
def test_a_run_that_blows_up(mode, periodic):
    """Fluid velocities that carry the nodes past the integers in one step: the
    run ends in an error or in values, and the next solver is none the worse."""
    for axis in range(3):
        s = solver(periodic, 0, mode=mode)
        n = s.n
        u = [np.full(n, 1e13 if a == axis else 0.0) for a in range(3)]
        s.set_state(np.ones(n), *u)
        print("axis %d, mode %d" % (axis, mode), flush=True)
        try:
            s.step(6)
            s.sync()
            s.membrane_nodes()
        except abi.LbfsError as e:
            assert "not finite" in str(e)
        s.close()
    s = solver((0, 0, 0))
    s.step(2)
    assert all(np.all(np.isfinite(v)) for v in s.get_state())
    s.close()
