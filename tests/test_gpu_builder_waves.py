"""Builder kernels that give each triangle or wall-adjacent cell a wave, on the
GPU against the oracle, bit for bit: bins of fewer and of many more triangles
than a wave has lanes, triangles in one bin and in hundreds, one and two
bodies, one and two levels, more triangles and wall-adjacent cells than the
launch has waves (16384)."""
import numpy as np
import pytest

from lbm3_amd import cases, geometry, lib
from tests.oracle_lib import OracleSim

pytestmark = pytest.mark.gpu

ARRAYS = ("shifter", "wallMap", "wallIndex", "wallData", "linkLength")


def _sphere(segments, size=24, levels=1):
    case, dom, _ = cases.sphere(2 * size, size, size, diameter=size / 4.0, center=(size / 2.0, size / 2.0, size / 2.0))
    if levels > 1:
        case.gridLevelCount = levels
        h = size / 4.0
        cases.add_refine_rule(case, 0, [size / 2.0 - h] * 3 + [size / 2.0 + h] * 3)
    return case, dom, [geometry.uv_sphere(size / 8.0, (size / 2.0,) * 3, *segments)]


def _two_bodies():
    case, dom, tris = _sphere((16, 32))
    return case, dom, tris + [geometry.box((30.3, 8.2, 7.6), (34.7, 12.9, 13.1))]


CASES = {
    "box of 12 triangles": lambda: (lambda c: (c[0], c[1], [geometry.box((8.3, 8.2, 7.6), (14.7, 12.9, 13.1))]))(_sphere((4, 8))),
    "8x16": lambda: _sphere((8, 16)),
    "120x240, most of them in each bin's reach": lambda: _sphere((120, 240), 16),
    "60x120 on two levels": lambda: _sphere((60, 120), levels=2),
    "two bodies": _two_bodies,
    "more items than waves": lambda: (lambda c: (c[0], c[1], [geometry.uv_sphere(33.0, (40.2, 40.1, 39.7), 100, 200)]))(
        _sphere((4, 8), 80)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_walls_and_links_equal_the_oracle(name):
    case, dom, tris = CASES[name]()
    o = OracleSim(case, dom, tris)
    s = lib.Sim(case, "f32")
    s.build(dom, tris)
    for level in range(case.gridLevelCount):
        for a in ARRAYS:
            assert np.array_equal(s.array(a, level), o.array(a, level)), (level, a)
        b, c = s.info(level).Bounds, o.info(level).Bounds
        assert [getattr(b, k) for k, _ in b._fields_] == [getattr(c, k) for k, _ in c._fields_]
    assert s.array("wallIndex", case.gridLevelCount - 1).size > (16384 if name == "more items than waves" else 0)
