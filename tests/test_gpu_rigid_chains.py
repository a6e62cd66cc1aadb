"""Whole-box pair sums (energies, forces, torques, virial) of molecules other
than one- and three-site ones against the oracle: 5, 8 and 16 atoms (a home
molecule of more than four takes several passes, and 64 near molecules of 16
fill a wave's atom list), alone and beside a one-site kind (molecules of unequal
length), more atom types than the table in LDS holds, exponents other than 12,
and counts on both sides of the line where a home molecule has one wave or four.

Bar: that of the three-site tests: energies 1e-11 relative, components 1e-9 of
the largest of their array.
"""
import numpy as np
import pytest

from gomc_amd.api import Box
from oracle.pyoracle import Oracle
from rigid_chains import chain_box, chain_kind

pytestmark = pytest.mark.gpu


def one_site(t):
    k = chain_kind(1, 1, first_type=t)
    k.charges = [0.0]
    return k


def mixed(a, n, m, edge, types, **kw):
    kinds = [chain_kind(a, types - 1), one_site(types - 1)]
    mk = np.random.default_rng(7).permutation([0] * n + [1] * m)
    return chain_box(kinds, mk, (edge,) * 3, types, **kw)


CASES = {
    "5_atoms_3_types": lambda: chain_box([chain_kind(5, 3)], [0] * 180, (26.0, 29.0, 24.0), 3),
    "16_atoms_10_types": lambda: chain_box([chain_kind(16, 10)], [0] * 90, (30.0,) * 3, 10),
    "16_atoms_dense": lambda: chain_box([chain_kind(16, 8)], [0] * 140, (27.0,) * 3, 8, rcut=13.0),
    "16_and_1": lambda: mixed(16, 40, 300, 34.0, 9),
    "8_and_1_mie": lambda: mixed(8, 60, 200, 30.0, 5, n_rep=[12.0, 14.0, 15.3, 12.0, 16.0]),
    "no_electrostatics": lambda: mixed(6, 60, 100, 28.0, 4, ewald=False, electrostatic=False),
    "one_wave_3100": lambda: mixed(16, 60, 3040, 55.0, 11),
    "one_wave_5_atoms": lambda: chain_box([chain_kind(5, 4)], [0] * 3100, (62.0, 60.0, 64.0), 4),
}


def near(a, b, tol=1e-9):
    a, b = np.asarray(a), np.asarray(b)
    assert np.abs(a - b).max() <= tol * max(np.abs(b).max(), 1e-300)


@pytest.mark.parametrize("name", CASES)
def test_pair_sums(name):
    s = CASES[name]()
    b, o = Box(s), Oracle(s, threads=8)
    for x, y in zip(b.box_inter(), o.box_inter()):
        assert abs(x - y) <= 1e-11 * abs(y)
    lj, real, fa, fm = b.box_force()
    olj, oreal, ofa, ofm = o.box_force()
    assert abs(lj - olj) <= 1e-11 * abs(olj) and abs(real - oreal) <= 1e-11 * abs(oreal)
    near(fa, ofa)
    near(fm, ofm)
    if s.ewald:
        ra, rm = b.box_force_recip()
        ora, orm = o.box_force_recip()
        near(ra, ora)
        near(rm, orm)
        near(b.torque(), o.torque())
    v, ov = b.virial(), o.virial()
    for key in ("inter", "real", "recip"):
        assert abs(v[key] - ov[key]) <= 1e-9 * np.abs(ov["tensor"]).max(), key
    near(v["tensor"], ov["tensor"])
    near(b.system_total(), o.system_total(), 1e-11)
    b.close()
    o.close()


@pytest.mark.parametrize("atoms", [2, 5, 16])
def test_host_moves(atoms):
    s = chain_box([chain_kind(atoms, 4)], [0] * 60, (26.0,) * 3, 4)
    b, o = Box(s), Oracle(s, threads=8)
    _, rec = b.run(200)
    _, orec = o.run(200, mode=0)
    assert np.array_equal(rec["acc"], orec["acc"])
    near(b.coords(), o.coords())
    b.close()
    o.close()
