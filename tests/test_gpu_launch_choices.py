"""The levels' own launch choices (nothing set) against lbm3_get_tune,
lbm3_set_tune, lbm3_autotune and a loaded checkpoint."""
import numpy as np
import pytest

from lbm3_amd import cases, lib

pytestmark = pytest.mark.gpu


def _sim(make, storage="f32"):
    case, dom, tris = make()
    s = lib.Sim(case, storage)
    s.build(dom, tris)
    s.init()
    return s


def _levels():
    return cases.multilevel_sphere(128, 64, 64, diameter_fine=24.0, seed=0)


def test_choices_reported_before_and_after_the_first_run():
    """A level of 64 to 256 MiB with open cells (they decide its LDS choice, and
    are classified by the first run)."""
    s = _sim(lambda: cases.sphere(96, 96, 96, diameter=24.0, center=(24.0, 48.0, 48.0), segments=(16, 32)))
    before = s.tune()
    s.run(2)
    assert s.tune() == before
    s.set_tune(*(before[k] for k in lib.Sim.TUNE))
    assert s.tune() == before
    s.run(2)
    assert s.tune() == before
    s.close()


def _turns(sims, steps=20, rounds=7):
    t = [[] for _ in sims]
    for _ in range(rounds):
        for k, s in enumerate(sims):
            t[k].append(s.run_timed(steps)[0])
    return [float(np.min(x)) for x in t]


def test_set_and_autotuned_choices_are_not_slower_on_three_levels():
    """Setting what is reported leaves every level its own choices, and the
    autotuner keeps them unless a set of choices is faster.  As one set for all
    levels they ran 6 to 11% slower; runs of one side differ by about 1%."""
    own, same, tuned = (_sim(_levels) for _ in range(3))
    for s in (own, same, tuned):
        s.run(4)
    t = same.tune()
    same.set_tune(*(t[k] for k in lib.Sim.TUNE))
    tuned.autotune(steps=3)
    a, b, c = _turns((own, same, tuned))
    print("three levels, ms per 20 steps: own %.3f, set as reported %.3f, autotuned %.3f" % (a, b, c))
    assert b < 1.04 * a and c < 1.04 * a
    for s in (own, same, tuned):
        s.close()


def test_a_loaded_x_face_split_changes_no_other_choice(tmp_path):
    """A checkpoint with a condition pending for the split layout: the loading
    simulation adopts the split, keeps its other choices and continues bit for bit."""
    make = lambda: cases.sphere(48, 24, 24, diameter=6.0, center=(14.0, 12.0, 12.0), segments=(16, 32))
    a, b = _sim(make), _sim(make)
    a.set_tune(40960, 0, 1, 8, 1)
    a.run(9)
    a.save_checkpoint(tmp_path / "c")
    a.run(6)
    own = b.tune()
    b.load_checkpoint(tmp_path / "c")
    assert b.tune() == dict(own, open_split=1)
    b.run(6)
    assert np.array_equal(a.macros(0), b.macros(0))
    # still the levels' own: another layout, and back by setting what is reported
    t = b.tune()
    b.set_tune(*(t[k] for k in lib.Sim.TUNE))
    assert b.tune() == t
    for s in (a, b):
        s.close()


@pytest.mark.parametrize("storage", ["f16", "bf16", "f16c"])
@pytest.mark.parametrize("layout", [(40960, 2, 1, 8, 0), (0, 3, 3, 1, 0), (0, 3, 1, 1, 3), (0, 2, 3, 16, 0)])
def test_rotor_choice_leaves_the_other_cells_of_16_bit_levels(layout, storage):
    """Whether the bulk kernel steps the rotor cells or a kernel of their own does,
    the cells that share no wave with them collide with the same arithmetic:
    after one step the same bits."""
    case, dom, statics, rotor, info = cases.rotor_duct(192, 24, 24, seed=1, levels=1, n_theta=128, n_axial=8)
    out = []
    for in_bulk in (0, 1):
        s = lib.Sim(case, storage)
        s.build(dom, statics)
        s.build_rotors([rotor])
        s.set_rotor(0, 0, info["omega"], info["axis"], info["origin"])
        s.init_fields(0, ((np.random.RandomState(5).rand(s.info(0).cellCount, 4) - 0.5) *
                          np.array([0.004, 0.04, 0.04, 0.04])).astype(np.float32))
        s.set_tune(*layout, in_bulk)
        s.run(1)
        kind = (s.array("cellRow", 0) & 0xFFFFFFFF).astype(np.uint32).view(np.int32)
        out.append(s.populations(0).view(np.uint16))
        shifter, row_i = s.array("shifter", 0), s.array("rowI", 0)
        s.close()
    a, b = out
    # cells (rows lie along x) more than a wave from the rotor's, and its slots
    head = np.maximum.accumulate(np.where(shifter >= 0, np.arange(kind.size), 0))
    x = row_i[shifter[head]] + np.arange(kind.size) - head
    rotor_x = x[kind == -4]
    far = (x > rotor_x.max() + 66) | (x < rotor_x.min() - 66)
    wave = np.arange(kind.size) // 64
    far &= ~np.isin(wave, np.unique(wave[kind == -4]))
    far &= (kind == -1) | (kind == -2) | (kind <= -5)
    assert far.sum() > 1000
    assert np.array_equal(a[:, far], b[:, far])
