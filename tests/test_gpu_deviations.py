"""The bulk kernel's collision on 16-bit deviations, on the GPU, against the same
run in FP64 storage.  One step from the same state moves a deviation by at most
one rounding of the storage (half a unit in the last place: 2^-11 of the value
for FP16, 2^-12 for f16c, 2^-8 for BF16) beyond what the start's own rounding
carries through one collision (norm at most 2 on the deviations), so three
roundings bound the 2-norm.  Cases: box edges (rows of 6 to 66 cells, images on
and off), reference velocities, both collision variants, forces, open faces."""
import numpy as np
import pytest

from lbm3_amd import cases, lib

pytestmark = pytest.mark.gpu

ULP = {"f16": 2.0 ** -11, "f16c": 2.0 ** -12, "bf16": 2.0 ** -8}


def _box(n, limiter=0.0, ref=(0.0, 0.0, 0.0)):
    case, dom, tris = cases.periodic_box(n, nu=0.03, limiter=limiter)
    case.storeRef[0], case.storeRef[1], case.storeRef[2] = ref
    return case, dom, tris


CASES = {
    "box 4": lambda: _box(4),
    "box 22 K17": lambda: _box(22, 0.1),
    "box 64 K17, moving reference": lambda: _box(64, 0.1, (0.05, -0.02, 0.03)),
    "box 30, moving reference": lambda: _box(30, 0.0, (0.05, 0.0, 0.0)),
    "forced duct": lambda: cases.channel(66, 14, 18, force=1e-4, nu=0.05),
    "sphere, open cells in the bulk kernel": lambda: cases.sphere(70, 34, 32, diameter=9.0, center=(20.0, 17.0, 16.0),
                                                                  segments=(16, 32)),
}


@pytest.mark.parametrize("storage", ["f16", "bf16", "f16c"])
@pytest.mark.parametrize("name", list(CASES))
def test_steps_stay_within_roundings_of_fp64(name, storage):
    case, dom, tris = CASES[name]()
    ref = np.array([case.storeRef[k] for k in range(3)])
    out = []
    for st in ("f64", storage):
        s = lib.Sim(case, st)
        s.build(dom, tris)
        n = s.info(0).cellCount
        f = (np.random.RandomState(1).rand(n, 4) - 0.5) * np.array([0.004, 0.02, 0.02, 0.02])
        f[:, 1:] += ref
        s.init_fields(0, f.astype(np.float32))
        fluid = s.array("wallMap", 0) != -3      # solid cells' slots are never stepped
        got = []
        for steps in (1, 1, 4):
            s.run(steps)
            got.append(s.macros(0)[fluid].astype(np.float64) - np.concatenate([[0.0], ref]))
        out.append(got)
        s.close()
    # deviations of the fields from the reference state; 27 populations average
    # their roundings, which the bound of three per step leaves out
    for k, steps in enumerate((1, 2, 6)):
        a, b = out[0][k], out[1][k]
        err = np.linalg.norm(b - a) / np.linalg.norm(a)
        print("%s %s after %d steps: %.2e of %.2e" % (name, storage, steps, err, 3 * (steps + 1) * ULP[storage]))
        assert err < 3 * (steps + 1) * ULP[storage]


@pytest.mark.parametrize("storage", ["f16", "bf16", "f16c"])
@pytest.mark.parametrize("limiter", [0.0, 0.1])
def test_the_reference_state_stays(storage, limiter):
    """A uniform flow at the reference velocity is all zero deviations (of either
    sign) and stays so exactly."""
    case, dom, tris = _box(18, limiter, (0.04, 0.01, -0.02))
    s = lib.Sim(case, storage)
    s.build(dom, tris)
    f = np.zeros((s.info(0).cellCount, 4), np.float32)
    f[:, 1:] = (0.04, 0.01, -0.02)
    s.init_fields(0, f)
    s.set_populations(0, np.zeros_like(s.populations(0)))
    s.run(8)
    assert not (s.populations(0).view(np.uint16) & 0x7FFF).any()
    s.close()
