"""One molecule's trial against totals of the whole box where the trial's
reciprocal blocks take one run of k-vectors, two and more (the line is 256
blocks of 128 k-vectors, 512 for molecules of more than four atoms), ragged at
the end, with and without the cell walk, and for molecules of 1 to 16 atoms.

Bar: 1e-11 of the largest term.  A trial's energies are differences of sums the
totals hold too; each sum of T terms is within about sqrt(T) roundings of 1.1e-16
of its largest partial sum, 1e-13 for the 1e6 (atom, k) and pair terms here, and
the totals' phases and erfc are good to some 1e-15 of a term.
"""
import numpy as np
import pytest

from gomc_amd import systems
from gomc_amd.api import Box
from rigid_chains import chain_box, chain_kind

pytestmark = pytest.mark.gpu


def check(s, m):
    b = Box(s)
    before = b.system_total()
    xyz = b.coords()
    at = slice(int(s.mol_start()[m]), int(s.mol_start()[m]) + b.mol_len(m))
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
    b.close()


def runs(b, atoms):
    return -(-(-(-b.nkvec // 128)) // (256 if atoms <= 4 else 512))


@pytest.mark.parametrize("n,rcut,want", [(216, 9.0, 1), (700, 5.2, 1), (700, 4.6, 1),
                                         (1000, 4.0, 2), (1000, 3.5, 3)])
def test_trial_equals_totals(n, rcut, want):
    s = systems.water_box(n, rcut=rcut, seed=11)
    b = Box(s)
    assert runs(b, 3) == want
    b.close()
    check(s, n // 3)


@pytest.mark.parametrize("atoms,n,edge,rcut,want", [
    (1, 200, 24.0, 8.0, 1), (2, 150, 24.0, 8.0, 1), (4, 100, 24.0, 8.0, 1), (5, 60, 24.0, 8.0, 1),
    (16, 40, 30.0, 8.0, 1), (16, 60, 42.0, 5.2, 1), (16, 60, 42.0, 4.3, 2)])
def test_other_lengths(atoms, n, edge, rcut, want):
    kind = chain_kind(atoms, 4)
    if atoms == 1:
        kind.charges = [0.25]
    s = chain_box([kind], [0] * n, (edge,) * 3, 4, rcut=rcut)
    b = Box(s)
    assert runs(b, atoms) == want
    b.close()
    check(s, n // 3)
