"""The two reconstructions of a face (faces whose lattice directions all lie
clearly on one side; faces with a direction in or near their plane, and
boundary faces) against the FP64 oracle, on meshes that hold one kind, the
other, and both: orthogonal cells (every interior face has directions in its
plane), cells jittered by 2e-3 (|e.n| on both sides of the tie band of
0.001 dt_f = 5e-4) and by 0.1."""
import numpy as np
import pytest

import cases
from lbfs_amd import abi
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lat_a,lat_o", cases.LAT_PAIRS)
@pytest.mark.parametrize("flags", [0, abi.FLAG_UPWIND_BAND])
@pytest.mark.parametrize("jitter,gamma,scale", [(0.0, 1.0, 1.0), (2e-3, 1.0, 1.0), (0.1, 0.4, 1.0), (0.1, 1.0, 4e-10)])
def test_face_classes(lat_a, lat_o, flags, jitter, gamma, scale):
    # (scale 4e-10: squared areas below 1e-36, where the normal's length comes
    # from the library's square root)
    n = (11, 9, 7)
    m = abi.HexMesh(*n, lengths=tuple(scale * k for k in n), periodic=(1, 0, 1), jitter=jitter, seed=6)
    visc = scale / 6.0
    s = abi.Solver(m, abi.make_params(lattice=lat_a, visc=visc, gamma=gamma, dt=0.25 * scale, flags=flags))
    o = orc.OracleFluid(m, lat_o, visc=visc, gamma=gamma, dt=0.25 * scale, flags=flags)
    st = cases.smooth_state(m, seed=15)
    s.set_state(*st)
    o.set_state(*st)
    fs, fo = s.face_flux().reshape(-1, 4) / scale ** 2, o.face_flux().reshape(-1, 4) / scale ** 2
    # 2e-7: a few single-precision roundings of the terms of a unit face's
    # momentum flux (|u| 0.01, drho 1e-3, tau Tx up to 0.03 with gamma 0.4)
    assert cases.rel_l2(fs[:, 0], fo[:, 0]) < 1e-5
    for v in range(1, 4):
        d = fs[:, v] - fo[:, v]
        assert np.sqrt(np.mean(d * d)) < 2e-7 / min(gamma, 1.0), (v, np.abs(d).max())
    s.close()
