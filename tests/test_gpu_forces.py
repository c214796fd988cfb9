"""The membrane forces in one launch against the separate passes (the named
stages of a step): the same bits, for node counts around the workgroups' size,
several membranes of different moduli, and nodes with more springs than lanes."""
import numpy as np
import pytest

import cases
from lbfs_amd import abi

pytestmark = pytest.mark.gpu


def bipyramid(n, center, r=4.0):
    """Two apexes over an n-gon: 4 n spring shares at each apex."""
    a = 2 * np.pi * np.arange(n) / n
    x = np.concatenate([np.stack([r * np.cos(a), r * np.sin(a), 0.2 * np.cos(3 * a)], 1), [[0, 0, 3.0], [0, 0, -3.0]]])
    k = np.arange(n)
    t = np.concatenate([np.stack([k, (k + 1) % n, 0 * k + n], 1), np.stack([(k + 1) % n, k, 0 * k + n + 1], 1)])
    return x + np.array(center), t.astype(np.int32)


def cells(kind):
    p = dict(abi.RBC_PARAMS, volume_ratio=0.95, local_bending_modulus=1e-3, viscosity=0.02)
    if kind == "fans":  # apexes of 4, 16, 17 and 40 shares; 3 to 12 nodes
        return [abi.Membrane(*bipyramid(n, (6 + 4 * i, 8, 8)), **p) for i, n in enumerate((3, 4, 5, 10))]
    if kind == "one":
        return [abi.Membrane(*abi.rbc(8, 9.0, center=(12, 8, 8)), **p)]  # 642 nodes: 20 workgroups and 2 nodes
    q = dict(p, shear_modulus=2e-3, mad_compat=1, spring_law=1)
    return [abi.Membrane(*abi.rbc(f, 4.0, center=(4 + 4 * i, 5 + 2 * i, 8)), **(q if i % 2 else p))
            for i, f in enumerate((1, 2, 4, 3, 2))]  # 12 to 162 nodes


@pytest.mark.parametrize("kind", ["one", "several", "fans"])
@pytest.mark.parametrize("mode", [0, 1, 2])
def test_one_launch_equals_separate_passes(kind, mode):
    outs = []
    for whole in (True, False):
        mesh = cases.channel_mesh(24, 16, 16, seed=31)
        s = abi.Solver(mesh, abi.make_params(visc=1.0 / 6.0, dt=0.25, body_force=(2e-5, 0.0, 0.0)))
        s.set_state(*cases.smooth_state(mesh, seed=31, amp=0.005))
        s.set_ibm_binned(mode)
        s.add_membranes(cells(kind), ibm_kernel=abi.IBM_COS4)
        if whole:
            s.step(5)
        else:
            for _ in range(5):
                for n in s.stage_names():
                    s.stage_run(n)
                s.stage_end_step()
        outs.append((np.concatenate(s.get_state()), *s.membrane_nodes(), s.membrane_globals(), s.cell_force()))
        s.close()
    assert np.abs(outs[0][3]).max() > 0
    for a, b in zip(*outs):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)
