"""Threads that read one simulation at the same time (its buffers kept between
calls, the calls outside the interpreter's lock): every read equals the same read
alone."""
import threading

import numpy as np
import pytest

from lbm3_amd import cases, lib

pytestmark = pytest.mark.gpu


def _together(reads, rounds=30):
    """Each read in a thread of its own, `rounds` times; the results that differ
    from the read alone."""
    want = [r() for r in reads]
    wrong, gate = [], threading.Barrier(len(reads))

    def loop(k):
        for n in range(rounds):
            gate.wait(timeout=60)
            try:
                if not np.array_equal(reads[k](), want[k]):
                    wrong.append((k, n))
            except Exception as e:      # a failed read must not leave the others at the barrier
                wrong.append((k, n, e))

    threads = [threading.Thread(target=loop, args=(k,)) for k in range(len(reads))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=90)
    return wrong


def test_fields_of_two_levels():
    case, dom, tris = cases.taylor_green(32, levels=2)
    s = lib.Sim(case, "f32")
    s.build(dom, tris)
    s.init()
    s.run(3)
    assert not _together([lambda: s.macros(0), lambda: s.macros(1), lambda: s.macros(0), lambda: s.macros(1)])
    s.close()


def test_rotor_forces_beside_the_energy():
    case, dom, statics, rotor, info = cases.rotor_duct(48, 24, 24, seed=1, levels=2, n_theta=128, n_axial=8)
    s = lib.Sim(case, "f32")
    s.build(dom, statics)
    s.build_rotors([rotor])
    for level in range(2):
        s.set_rotor(level, 0, info["omega"], info["axis"], info["origin"])
    s.init()
    s.run(5)
    assert not _together([lambda: s.rotor_forces(0, 0), lambda: s.rotor_forces(1, 0), lambda: np.array([s.kinetic_energy()])])
    s.close()
