"""The tile spreading at the edges of its rules, against the per-node spreading
(the same 64-bit sums, so the same bits): boxes shorter than a stencil, where a
node reaches a tile through several of its periodic images; tiles of one cell
and so many of them that the smaller workgroups run; forces whose terms leave
the range of the short conversion."""
import numpy as np
import pytest

import cases
from lbfs_amd import abi

pytestmark = pytest.mark.gpu

MODULI = ("shear_modulus", "volume_modulus", "local_area_modulus", "global_area_modulus", "global_bending_modulus",
          "local_bending_modulus")


def run(mode, n, tile, kernel, steps, scale=1.0, d0=6.0):
    mesh = abi.HexMesh(*n, periodic=(1, 1, 1), seed=3)
    s = abi.Solver(mesh, abi.make_params(visc=1.0 / 6.0, dt=0.25, tile=tile))
    s.set_state(*cases.smooth_state(mesh, seed=3, amp=0.005))
    s.set_ibm_binned(mode)
    x, t = abi.rbc(4, d0, center=tuple(0.5 * k for k in n))
    # forces are linear in the moduli
    p = dict(abi.RBC_PARAMS, volume_ratio=0.95, viscosity=0.0)
    p.update({k: scale * p[k] for k in MODULI})
    s.add_membranes([abi.Membrane(x, t, **p)], ibm_kernel=kernel)
    s.step(steps)
    X, U, F = s.membrane_nodes()
    out = (np.concatenate(s.get_state()), s.cell_force(), X, F)
    s.close()
    return out


@pytest.mark.parametrize("kernel", [abi.IBM_COS4, abi.IBM_LINEAR2, abi.IBM_LAGRANGE4])
@pytest.mark.parametrize("n,tile", [
    ((1, 16, 12), (0, 0, 0)),    # four images along x
    ((2, 3, 16), (0, 0, 0)),     # three and two
    ((9, 12, 11), (8, 8, 8)),    # both ends of a tile that spans most of the box
    ((10, 9, 11), (8, 8, 8)),
    ((24, 16, 16), (1, 1, 1)),   # 6144 tiles, 64 neighbours each
    ((40, 32, 32), (4, 2, 1)),   # 5120
])
def test_tile_spreading_equals_per_node(n, tile, kernel):
    a = run(0, n, tile, kernel, 4)
    b = run(1, n, tile, kernel, 4)
    assert np.abs(a[1]).max() > 0 and all(np.all(np.isfinite(v)) for v in a)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("mode", [1, 2])
def test_terms_beyond_the_short_conversion(mode):
    n = (16, 16, 16)
    f1 = np.abs(run(0, n, (0, 0, 0), abi.IBM_COS4, 1)[3]).max()
    # weights reach 1/8: the largest terms lie between 2^11 and their limit 2^12
    a, b = (run(m, n, (0, 0, 0), abi.IBM_COS4, 1, scale=28000.0 / f1) for m in (0, mode))
    assert 2048 < 0.1 * np.abs(a[3]).max() < 4096
    assert np.all(np.isfinite(a[1])) and np.array_equal(a[3], b[3]) and np.array_equal(a[1], b[1])
