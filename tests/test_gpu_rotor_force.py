"""The rotor force sums on the device against the oracle's, for rotors of one
marked block's worth of force cells up to several blocks of threads."""
import numpy as np
import pytest

from lbm3_amd import cases, geometry, lib
from lbm3_amd import ctypes_defs as T
from tests.oracle_lib import OracleSim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("radius,length", [(1.2, 1.0), (4.0, 3.0), (8.5, 8.0)])
def test_rotor_forces_equal_the_oracle(radius, length):
    case, dom, _ = cases.periodic_box(24, u=(0.01, 0.0, 0.005))
    case.trackRotorForce = 1
    rot = geometry.rotor(3, radius, 0.4, 20.0, length, (0.3, -0.2, 0.1), axis=2, n_theta=96, n_axial=6)
    o, g = OracleSim(case, dom, [], double=True), lib.Sim(case, "f64")
    g.build(dom, [])
    for s in (o, g):
        s.build_rotors([rot])
        s.set_rotor(0, 0, 0.01, T.AXIS_Z, (0.3, -0.2, 0.1))
        s.init()
    o.run(12)
    g.run(12)
    want, got = o.rotor_forces(0, 0), g.rotor_forces(0, 0)
    assert np.abs(want).max() > 0
    # FP64 sums of 27 values per marked block in another order, on fields 1e-10 apart
    assert np.abs(got - want).max() < 1e-9 * np.abs(want).max()
    g.reset_wall_forces()
    assert not g.rotor_forces(0, 0).any()
    g.close()
