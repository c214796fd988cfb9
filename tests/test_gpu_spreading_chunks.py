"""The tile spreading where a tile looks at many chunks of candidate nodes, most
of them out of its reach, so that its wavefronts drift apart between chunks:
equal bit for bit to the per-node spreading at every step."""
import numpy as np
import pytest

import cases
from lbfs_amd import abi

pytestmark = pytest.mark.gpu


def run(mode, n, tile, freq, kernel, steps):
    mesh = abi.HexMesh(*n, periodic=(1, 1, 1), seed=5)
    s = abi.Solver(mesh, abi.make_params(visc=1.0 / 6.0, dt=0.25, tile=tile))
    s.set_state(*cases.smooth_state(mesh, seed=5, amp=0.005))
    s.set_ibm_binned(mode)
    x, t = abi.rbc(freq, 6.0, center=tuple(0.5 * k for k in n))
    s.add_membranes([abi.Membrane(x, t, **dict(abi.RBC_PARAMS, volume_ratio=0.95, viscosity=0.0))], ibm_kernel=kernel)
    out = []
    for _ in range(steps):
        s.step(1)
        out.append(s.cell_force())
    out += list(s.get_state()) + list(s.membrane_nodes())
    s.close()
    return out


@pytest.mark.parametrize("n,tile,freq", [
    ((24, 16, 16), (8, 8, 8), 16),   # chunks of 512: 2562 nodes, most of them in the overflow list
    ((40, 32, 32), (4, 2, 1), 16),   # of 256 (5120 tiles)
    ((2, 3, 16), (0, 0, 0), 6),      # of 56 (nine images kept)
    ((1, 16, 12), (0, 0, 0), 8),     # of 128
])
@pytest.mark.parametrize("kernel", [abi.IBM_COS4, abi.IBM_LINEAR2])
def test_many_chunks_equal_per_node(n, tile, freq, kernel):
    a = run(0, n, tile, freq, kernel, 6)
    b = run(1, n, tile, freq, kernel, 6)
    assert np.abs(a[0]).max() > 0 and all(np.all(np.isfinite(v)) for v in a)
    for x, y in zip(a, b):
        assert np.array_equal(x, y)
