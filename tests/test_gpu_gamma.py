"""Preconditioning factors beyond single precision (the limit in which only the
linear terms are left) against the FP64 oracle."""
import numpy as np
import pytest

import cases
from lbfs_amd import abi
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lat_a,lat_o", cases.LAT_PAIRS)
@pytest.mark.parametrize("gamma", [1e37, 1e39, float("inf")])
def test_large_gamma(lat_a, lat_o, gamma):
    n = (24, 20, 1) if lat_a == abi.D2Q9 else (11, 9, 7)
    m = abi.HexMesh(*n, periodic=(1, 1, 1), jitter=0.1, seed=6)
    s = abi.Solver(m, abi.make_params(lattice=lat_a, visc=1.0 / 6.0, gamma=gamma, dt=0.25))
    o = orc.OracleFluid(m, lat_o, visc=1.0 / 6.0, gamma=gamma, dt=0.25)
    st = cases.smooth_state(m, seed=15)
    s.set_state(*st)
    o.set_state(*st)
    fs, fo = s.face_flux().reshape(-1, 4), o.face_flux().reshape(-1, 4)
    # (as for the finite factors: a few single-precision roundings of a unit
    # face's momentum flux)
    assert cases.rel_l2(fs[:, 0], fo[:, 0]) < 1e-5
    d = fs[:, 1:] - fo[:, 1:]
    assert np.sqrt(np.mean(d * d)) < 2e-7, np.abs(d).max()
    s.step(5)
    assert all(np.all(np.isfinite(v)) for v in s.get_state())
    s.close()
