"""The transposes of the two face reconstructions (faces clear of every lattice
direction; faces with a direction in or near their plane, and boundary faces)
against directional differences of the FP64 oracle, on meshes that hold both
kinds and mostly one, with face lists shorter than one chunk, ending just past
one, and of tiles with two cells a thread."""
import numpy as np
import pytest

import cases
from lbfs_amd import abi
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

VISC, DT, STEPS = 1.0 / 6.0, 0.25, 4


@pytest.mark.parametrize("lat_a,lat_o", cases.LAT_PAIRS)
@pytest.mark.parametrize("jitter", [2e-3, 0.1])
@pytest.mark.parametrize("tile,threads", [((3, 5, 4), 256), ((8, 6, 3), 512), ((8, 8, 15), 512)])
@pytest.mark.parametrize("flags", [0, abi.FLAG_GHOST_FACE_GRAD])
def test_state_adjoint_of_face_classes(lat_a, lat_o, jitter, tile, threads, flags):
    if lat_a == abi.D2Q9:
        mesh = abi.HexMesh(19, 13, 1, periodic=(1, 0, 1), jitter=jitter, seed=5)
    else:
        mesh = cases.channel_mesh(11, 9, 15, jitter=jitter, seed=5)
    st = cases.smooth_state(mesh, seed=5, amp=0.005)
    rng = np.random.default_rng(7)
    c = rng.standard_normal((mesh.n_cells, 4))
    v = 1e-3 * rng.standard_normal((mesh.n_cells, 4))
    if lat_a == abi.D2Q9:
        c[:, 3] = v[:, 3] = 0.0
    s = abi.Solver(mesh, abi.make_params(lattice=lat_a, visc=VISC, dt=DT, flags=flags, tile=tile,
                                         block_threads=threads))
    s.set_state(*st)
    s.adjoint_forward(STEPS, 3)
    ad = s.adjoint_backward(lam_state=c)["state0"] * v
    s.close()

    def loss(eps):
        o = orc.OracleFluid(mesh, lat_o, visc=VISC, dt=DT, flags=flags)
        o.set_state(*(st[k] + eps * v[:, k] for k in range(4)))
        o.step(STEPS)
        return float(np.sum(c * np.stack(o.state(), axis=1)))

    fd = (loss(1e-3) - loss(-1e-3)) / 2e-3
    # 1e-5 of the terms' root sum of squares: each term carries the roundings of
    # some 10 single-precision sums a step (6e-8 each), of independent sign
    # over the cells; the differences' own error is below 1e-8 of it
    assert abs(ad.sum() - fd) < 1e-5 * np.sqrt(np.sum(ad * ad)), (ad.sum(), fd)


@pytest.mark.parametrize("size,periodic", [((2, 7, 2), (1, 0, 1)), ((2, 2, 2), (1, 1, 1)), ((5, 1, 4), (1, 1, 1))])
def test_state_adjoint_of_repeated_neighbours(size, periodic):
    """Two layers and one between periodic sides: a cell meets a neighbour, or
    itself, through two faces."""
    mesh = abi.HexMesh(*size, periodic=periodic, jitter=0.1, seed=3)
    st = cases.smooth_state(mesh, seed=6, amp=0.005)
    rng = np.random.default_rng(8)
    c = rng.standard_normal((mesh.n_cells, 4))
    v = 1e-3 * rng.standard_normal((mesh.n_cells, 4))
    s = abi.Solver(mesh, abi.make_params(lattice=abi.D3Q19, visc=VISC, dt=DT))
    s.set_state(*st)
    s.adjoint_forward(STEPS, 3)
    ad = s.adjoint_backward(lam_state=c)["state0"] * v
    s.close()

    def loss(eps):
        o = orc.OracleFluid(mesh, orc.OR_D3Q19, visc=VISC, dt=DT)
        o.set_state(*(st[k] + eps * v[:, k] for k in range(4)))
        o.step(STEPS)
        return float(np.sum(c * np.stack(o.state(), axis=1)))

    fd = (loss(1e-3) - loss(-1e-3)) / 2e-3
    assert abs(ad.sum() - fd) < 1e-5 * np.sqrt(np.sum(ad * ad)), (ad.sum(), fd)  # (as above)
