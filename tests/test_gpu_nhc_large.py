"""The Nose-Hoover chain's share of a step: two calls of the chain in one launch
(steps that sample nothing) against one call per launch (a replayed graph), and
what the thermostat costs a large system."""
import time

import numpy as np
import pytest

from thrid_amd import md, systems

pytestmark = pytest.mark.gpu


def _context(s, v0):
    from thrid_amd.pgk import ForceContext
    ij, d, gs = md.rigid_constraints(s)
    c = ForceContext(s, "mixed")
    c.md_setup(s["mass"], ij, d, gs, 1.0)
    c.md_set_velocities(v0)
    return c


# the mixed form's sums are exact, and both ways run the same chain on the same
# records: bit for bit
def test_both_calls_in_one_launch():
    s = systems.water_box()
    v0 = md.maxwell_boltzmann(s, 300.0, seed=6)
    out = []
    for graphs in (False, True):
        c = _context(s, v0)
        c.md_nhc(330.0, tfreq=0.01, nfree=2 * s["natom"])
        c.md_use_graphs(graphs, graphs)
        c.md_run(30, 100, s["rcut_book"], 30)
        out.append(c.md_state() + tuple(np.ravel(x) for x in c.md_nhc_state()))
        c.close()
    for a, b in zip(*out):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)


def test_thermostat_does_not_grow_with_the_system():
    """A step of 300,000 atoms with the chain takes the records' pass and two
    calls more, some 21 us; a chain that waits for every block took 90."""
    nmol = 100000
    box = (nmol / 0.0334) ** (1.0 / 3.0)
    s = systems.water_box(box=box, nmol=nmol, rcut=10.0, rcut_book=11.0, alpha=0.3,
                          nfft=(144, 144, 144))
    c = _context(s, md.maxwell_boltzmann(s, 10.0, seed=1))

    def step_us():
        best = np.inf
        for _ in range(3):
            c.md_run(5, 1000, s["rcut_book"], 5)
            t = time.perf_counter()
            c.md_run(40, 1000, s["rcut_book"], 40)
            best = min(best, (time.perf_counter() - t) / 40 * 1e6)
        return best
    plain = step_us()
    c.md_nhc(300.0, tfreq=0.01, nfree=2 * s["natom"])
    chain = step_us()
    c.close()
    assert chain - plain < 50.0
