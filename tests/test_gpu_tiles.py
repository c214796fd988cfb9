"""The tile layout's slot patterns and halos: whole steps with the tile chosen
by the mesh's size equal the two-pass step on other tiles bit for bit, on
meshes whose halos are ragged, meet walls on every side, wrap onto the tile
itself (one and two layers), or have no logical numbering (whose tiles may
be too large for the fused pass, and then run the two passes)."""
import numpy as np
import pytest

import cases
from lbfs_amd import abi

pytestmark = pytest.mark.gpu


def renumbered(m, seed):
    """The mesh with its cells in random order and no logical structure."""
    p = np.random.default_rng(seed).permutation(m.n_cells).astype(np.int32)
    m.owner = p[m.owner].astype(np.int32)
    m.neighbour = p[m.neighbour].astype(np.int32)
    m.nx = m.ny = m.nz = 0
    return m, p


@pytest.mark.parametrize("size,periodic,tile,threads", [
    ((3, 5, 4), (0, 0, 0), (2, 2, 2), 256),       # one default tile and ragged ones, walls all round
    ((9, 5, 13), (1, 0, 1), (8, 8, 8), 512),      # the second halo reaches around the box
    ((2, 2, 2), (1, 1, 1), (1, 1, 1), 256),       # every neighbour twice
    ((17, 1, 9), (1, 1, 0), (4, 1, 4), 256),      # one layer: a cell is its own neighbour
    ((33, 19, 21), (1, 0, 0), (16, 8, 4), 512),   # ragged 8x4x4 default tiles
])
@pytest.mark.parametrize("ts", [0, abi.TS_MIN])
@pytest.mark.parametrize("logical", [True, False])
def test_default_tiles_equal_two_passes(size, periodic, tile, threads, ts, logical):
    m = abi.HexMesh(*size, periodic=periodic, jitter=0.1, seed=4)
    st = cases.smooth_state(m, seed=21)
    if not logical:
        m, p = renumbered(m, 8)
        inv = np.argsort(p)
        st = tuple(a[inv] for a in st)
    outs = []
    for fused, t, nt in ((True, (0, 0, 0), 0), (False, tile, threads)):
        s = abi.Solver(m, abi.make_params(lattice=abi.D3Q19, visc=1.0 / 6.0, dt=0.25, body_force=(2e-5, 0.0, 0.0),
                                          time_stepping=ts, max_velocity=0.02 if ts else 0.0, tile=t,
                                          block_threads=nt))
        if not fused:
            s.set_fused(False)
        s.set_state(*st)
        s.step(5)
        outs.append(np.concatenate(s.get_state()))
        s.close()
    assert np.all(np.isfinite(outs[0]))
    assert np.array_equal(outs[0], outs[1])
