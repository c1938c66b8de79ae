"""Periodic ghosts stepped by their source cells (one launch per step) against
the copy after every step, on the GPU: the same populations bit for bit.  A
captured step (run_graph) keeps the copy, so a replayed run is the copy path."""
import ctypes

import numpy as np
import pytest

from lbm3_amd import cases, lib

pytestmark = pytest.mark.gpu


def _make(case, dom, tris, storage, seed):
    s = lib.Sim(case, storage)
    s.build(dom, tris)
    n = s.info(0).cellCount
    r = np.random.RandomState(seed)
    # ghosts hold values of their own at the start, unlike their sources'
    f = (r.rand(n, 4).astype(np.float32) - 0.5) * np.array([0.002, 0.04, 0.04, 0.04], np.float32)
    s.init_fields(0, f)
    return s


BOXES = {
    "cube 4": lambda: cases.periodic_box(4),           # every cell a source of several ghosts
    "cube 14": lambda: cases.periodic_box(14),
    "cube 30 K17": lambda: cases.periodic_box(30, nu=0.02, limiter=0.1),
    "cube 62": lambda: cases.periodic_box(62),         # rows of a whole wave
    "duct": lambda: cases.channel(20, 12, 10),         # open cells beside the ghosts
    "plane channel": lambda: cases.channel(26, 8, 18, periodic_z=True),
}


def _sources(s):
    """Cells whose ghosts the bulk kernel steps; 0: the ghosts are copied."""
    return int(np.unpackbits(s.array("imageSources", 0).view(np.uint8)).sum())


@pytest.mark.parametrize("storage", ["f32", "f64", "f16", "bf16", "f16c"])
@pytest.mark.parametrize("box", list(BOXES))
def test_images_equal_the_copy(box, storage):
    a, b = (_make(*BOXES[box](), storage, 3) for _ in range(2))
    for steps in (1, 2, 5, 4):
        a.run(steps)
        assert _sources(a) == len(np.unique(a.array("periodicSource", 0)))
        b.run_graph(steps)
        got, last = a.populations(0), b.populations(0)
        assert got.tobytes() == last.tobytes(), (steps, np.argwhere(got.view(np.uint8) != last.view(np.uint8))[:4])
    a.run(3)
    b.run(3)
    assert a.macros(0).tobytes() == b.macros(0).tobytes()
    assert a.kinetic_energy() == b.kinetic_energy()


def test_images_with_open_cells_in_the_bulk_kernel():
    """Open cells completed by the bulk kernel (group width 1) beside ghosts."""
    sims = []
    for group in (1, 8):
        s = _make(*BOXES["duct"](), "f32", 5)
        s.run(1)
        s.set_tune(0, 2, 1, group)
        s.run(12)
        assert (_sources(s) > 0) == (group == 1)    # a ghost in a group is another kernel's
        sims.append(s)
    assert sims[0].populations(0).tobytes() == sims[1].populations(0).tobytes()


def test_images_checkpoint_and_graph(tmp_path):
    """Stale ghosts are copied before a checkpoint is written and before a capture."""
    a, b = (_make(*BOXES["cube 14"](), "f32", 9) for _ in range(2))
    a.run(5)
    b.run(5)
    assert _sources(a) > 0
    a.save_checkpoint(tmp_path / "c")
    a.run(4)
    a.run_graph(7)
    a.run(3)
    b.run(14)
    assert a.populations(0).tobytes() == b.populations(0).tobytes()
    a.load_checkpoint(tmp_path / "c")
    a.run(14)
    assert a.populations(0).tobytes() == b.populations(0).tobytes()


@pytest.mark.parametrize("n", [4, 6, 18, 30])
def test_short_rows_equal_the_oracle(n):
    """Rows of 6 to 32 cells (several to a wave, the table's padding within
    reach of the last wave) in FP64 against the oracle, ghosts included."""
    from tests.helpers import rel_max
    from tests.oracle_lib import OracleSim
    case, dom, tris = cases.periodic_box(n, u=(0.02, 0.01, -0.005))
    o = OracleSim(case, dom, tris, double=True)
    s = lib.Sim(case, "f64")
    s.build(dom, tris)
    f = (np.random.RandomState(n).rand(s.info(0).cellCount, 4) - 0.5) * np.array([0.002, 0.04, 0.04, 0.04])
    o.init_fields(0, f.astype(np.float32))
    s.init_fields(0, f.astype(np.float32))
    o.run(21)
    s.run(21)
    assert _sources(s) > 0
    a, b = o.macros(), s.macros(0)
    assert max(rel_max(1 + b[:, 0], 1 + a[:, 0]), rel_max(b[:, 1:], a[:, 1:])) < 1e-10


@pytest.mark.parametrize("storage", ["f32", "f16"])
@pytest.mark.parametrize("dims", [(24, 14, 12), (48, 24, 24), (70, 34, 32)])
def test_default_choices_equal_the_side_stream_kernels(dims, storage):
    """The one-launch default (open and wall cells in the bulk kernel's launch),
    also on the smallest boxes, against the kernels of their own: same bits."""
    case, dom, tris = cases.sphere(*dims, diameter=dims[1] / 4.0, center=(dims[0] / 4.0, dims[1] / 2.0, dims[2] / 2.0),
                                   segments=(16, 32))
    out = []
    for chosen in (None, (40960, 2, 1, 8)):
        s = lib.Sim(case, storage)
        s.build(dom, tris)
        s.init()
        if chosen:
            s.set_tune(*chosen)
        s.run(25)
        assert (s.cell_kinds(0)["open_in_bulk"] > 0) == (chosen is None)
        out.append((s.populations(0).tobytes(), s.wall_forces(0).tobytes()))
    assert out[0] == out[1]


def _same(a, b):
    return a.tobytes() == b.tobytes()


class _Kept:
    """The simulation's FP32 populations through their address (lbm3_device_array),
    copied on a stream other than the simulation's."""

    def __init__(self, s):
        L = lib.load()
        self.copy = L.hipMemcpy     # of the runtime the library itself uses
        ptr, n, tile, size = ctypes.c_void_p(), ctypes.c_longlong(), ctypes.c_int(), ctypes.c_int()
        lib.check(L.lbm3_device_array(s.h, 0, b"f", ctypes.byref(ptr), ctypes.byref(n)))
        lib.check(L.lbm3_population_layout(s.h, ctypes.byref(tile), ctypes.byref(size)))
        self.ptr, self.cells = ptr, s.info(0).cellCount
        self.shape = (n.value // (27 * tile.value), 27, tile.value)

    def _copy(self, dst, src, host, kind):
        assert self.copy(dst, src, ctypes.c_size_t(host.nbytes), kind) == 0

    def read(self):
        t = np.empty(self.shape, np.float32)
        self._copy(ctypes.c_void_p(t.ctypes.data), self.ptr, t, 2)
        return np.ascontiguousarray(t.transpose(1, 0, 2).reshape(27, -1)[:, :self.cells])

    def write(self, planes):
        t = np.zeros((27, self.shape[0] * self.shape[2]), np.float32)
        t[:, :self.cells] = planes
        t = np.ascontiguousarray(t.reshape(27, self.shape[0], self.shape[2]).transpose(1, 0, 2))
        self._copy(self.ptr, ctypes.c_void_p(t.ctypes.data), t, 1)


@pytest.mark.parametrize("box", ["cube 14", "cube 30 K17", "cube 62"])
def test_a_kept_address_sees_and_sets_the_ghosts(box):
    """The populations' address taken once: whatever call stepped, the ghosts are
    their sources' when it is waited for, and what is written there is what the
    next step takes (a simulation that gets the same state by upload)."""
    a, b = (_make(*BOXES[box](), "f32", 4) for _ in range(2))
    a.run(4)
    a.sync()
    f = _Kept(a)
    first = f.read()
    b.run_graph(4)
    assert _same(first, b.populations(0))
    ghosts = a.array("periodicIndex", 0)
    assert _sources(a) > 0
    for k, step in enumerate((lambda s: s.run(3), lambda s: s.run_graph(5), lambda s: s.run_timed(2, kernel_events=False),
                              lambda s: s.run(1))):
        step(a)
        a.sync()
        now = f.read()
        b.run_graph((3, 5, 2, 1)[k])
        assert _same(now, b.populations(0)), k
        # the ghosts get other values through the address
        now[:, ghosts[::3]] *= np.float32(1.25)
        f.write(now)
        b.set_populations(0, now)
    a.run(2)
    b.run_graph(2)
    assert _same(a.populations(0), b.populations(0))
