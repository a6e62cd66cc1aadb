"""One molecule's trial against totals of the whole box where the trial's
reciprocal blocks take one run of k-vectors, two and more (the line is 128
blocks of 128 k-vectors), ragged at the end, and with and without the cell walk.

Bar: 1e-11 of the largest term.  A trial's energies are differences of sums the
totals hold too; each sum of T terms is within about sqrt(T) roundings of 1.1e-16
of its largest partial sum, 1e-13 for the 1e6 (atom, k) and pair terms here, and
the totals' phases and erfc are good to some 1e-15 of a term.
"""
import numpy as np
import pytest

from gomc_amd import systems
from gomc_amd.api import Box

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,rcut,runs", [(216, 9.0, 1), (700, 5.2, 1), (700, 4.6, 2),
                                         (1000, 4.0, 3)])
def test_trial_equals_totals(n, rcut, runs):
    s = systems.water_box(n, rcut=rcut, seed=11)
    b = Box(s)
    assert -(-(-(-b.nkvec // 128)) // 128) == runs
    before = b.system_total()
    xyz = b.coords()
    m = n // 3
    at = slice(3 * m, 3 * m + 3)
    new = np.mod(xyz[at] + [0.21, -0.17, 0.3], b.dims()[:3])
    lj, real, recip, overlap = b.mol_trial(m, new)
    moved = xyz.copy()
    moved[at] = new
    b.set_coords(moved)
    after = b.system_total()
    scale = np.abs(np.concatenate([before, after])).max()
    assert overlap == 0.0
    assert abs(lj - (after[0] - before[0])) <= 1e-11 * scale
    assert abs(real - (after[2] - before[2])) <= 1e-11 * scale
    assert abs(recip - after[3]) <= 1e-11 * scale
