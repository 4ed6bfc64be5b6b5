"""Triangle groups (rigid water): ordinary displacements, and ones comparable
to a bond, whose sweeps start far from the constraints."""
import numpy as np
import pytest

from thrid_amd import md
from helpers import water648
import md_reference

pytestmark = pytest.mark.gpu


# 300 K: a separation's projection on the old one changes by 0.1 % at most;
# 60000 K: by a quarter (checked below)
@pytest.mark.parametrize("temperature,far", [(300.0, False), (60000.0, True)])
def test_triangle_sweeps_match_reference(oracle_mod, temperature, far):
    from thrid_amd.pgk import ForceContext
    s = water648()
    ij, d, gs = md.rigid_constraints(s)
    v0 = md.maxwell_boltzmann(s, temperature, seed=21)
    c = ForceContext(s, "fp64")
    c.md_setup(s["mass"], ij, d, gs, 1.0)
    c.md_set_velocities(v0)
    c.md_run(1, 20, s["rcut_book"], 1)
    p, v = c.md_state()
    c.close()
    rp, rv, _ = md_reference.run(oracle_mod.Oracle(s), s, v0, ij, d, gs, 1.0, 1)
    i, j = ij[:, 0] - 1, ij[:, 1] - 1
    old = s["pos"][i] - s["pos"][j]
    change = np.abs(((rp[i] - rp[j]) * old).sum(1) / (old * old).sum(1) - 1.0)
    assert (change.max() > 0.05) == far
    # both stop within 1e-10 d^2 of the constraint: 1e-9 leaves room for one
    # sweep more or less; the velocities carry that displacement over 1 fs
    assert np.max(np.abs(p - rp)) < 1e-9
    assert np.max(np.abs(v - rv)) < 1e-9 * max(1.0, np.max(np.abs(rv)))
