"""The pair search on both sides of the box width at which its minimum image
rounds differently (twice the cutoff), with atoms half a box apart, outside
the box and with more exclusions than are held in registers."""
import numpy as np
import pytest

from helpers import pairs_from_csr, water648

pytestmark = pytest.mark.gpu


def _star_exclusions(n):
    """1-based CSR, partners j > i: atom 1 excludes 2 .. 30, every third atom
    its two followers; an atom with none holds a single 0."""
    rows = [[] for _ in range(n)]
    rows[0] = list(range(2, 31))
    for i in range(30, n - 2, 3):
        rows[i] = [i + 2, i + 3]
    idx, lst = np.zeros(n + 1, np.int32), []
    for i in range(n):
        idx[i] = len(lst) + 1
        lst += rows[i] or [0]
    idx[n] = len(lst) + 1
    return idx, np.array(lst, np.int32)


# box 18.64: twice the cutoff is below it at 3 and 9.3 (the search's rounding
# to even), at it at 9.32 (the reference's half away); 9.35 is refused
@pytest.mark.parametrize("rcut_book", [3.0, 9.3, 9.32, 9.35])
@pytest.mark.parametrize("lattice", [False, True])
def test_pair_set(oracle_mod, rcut_book, lattice):
    from thrid_amd.pgk import ForceContext, PgkError
    s = water648()
    n = s["natom"]
    pos = s["pos"].copy()
    if lattice:   # pairs at exactly a half, and three halves, of the box
        k = np.arange(n)
        grid = np.stack([k % 8, (k // 8) % 8, (k // 64) % 8], 1) * (s["box"][0] / 8)
        pos = grid + 0.01 * (k // 512)[:, None]
    pos[::5] += np.asarray(s["box"]) * np.array([1.0, 2.0, 0.0])
    s = dict(s, pos=pos)
    excl = _star_exclusions(n)
    o = oracle_mod.Oracle(s, excl=excl)
    idx, lst = o.mklist(rcut_book, 0)
    want = pairs_from_csr(idx, lst, n)
    c = ForceContext(s, "fp64", excl=excl)
    if 2 * rcut_book > s["box"][0]:
        with pytest.raises(PgkError, match="exceeds half the box"):
            c.mklist(rcut_book)
        return
    c.mklist(rcut_book)
    got = c.list_pairs()
    assert len(want) > 0 and np.array_equal(got, want)
    c.close()
