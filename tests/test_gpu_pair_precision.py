"""The FP64 pair terms themselves, one pair at a time, against extended
precision: an atom at rest and trial positions or a second atom along x, at
distances of 24 bits whose squares are exact.

Bars, with u = 2^-53 and h half the repulsion exponent.  LJ, against the larger of
its two parts: x = sigma^2 / r^2 carries one rounding (taken as 1.1 u, since it is a
corrected product, not a division), the repulsion x^h h times that and 2 u of pow
(for h = 6 the square of the attraction, 2 x 5.3 u + u), the attraction x^3 3.3 u +
2 u, their difference and the factor epsilon one each:
u (max(1.1 h + 2, 12) + 5.3 + 2).

Coulomb: r = d and alpha r carry one rounding each, which erfc multiplies by
2 x^2, 23 at the cutoff; libm's erfc, 1 / r and the products add a few.  These
roundings have no preferred sign: over 1600 distances the mean of the errors, each
below 1.6e-15 in the mean square (23 u / sqrt(3)), is within 1.2e-16 (three
standard deviations) of 0.
"""
import ctypes

import numpy as np
import pytest

from gomc_amd import systems
from gomc_amd.api import Box

pytestmark = pytest.mark.gpu

U = 2.0 ** -53
L, RC, TOL = 48.0, 10.0, 1e-5


def two_atoms(n_rep, charge=0.0):
    kinds = [systems.MolKind("A", [0], [charge], np.zeros((1, 3))),
             systems.MolKind("B", [1], [-charge], np.zeros((1, 3)))]
    xyz = np.array([[16.0, 24.0, 24.0], [20.0, 24.0, 24.0]])
    return systems.System(box=(L,) * 3, temperature=300.0, rcut=RC, rcut_low=0.5, rcut_coulomb=RC,
                          tolerance=TOL, kinds=kinds, mol_kind=np.array([0, 1], np.int32), xyz=xyz,
                          sigma=[3.166, 2.9], epsilon=[78.2, 61.7], n_rep=[n_rep] * 2, lrc=False)


def distances(n, lo=2.0, hi=9.9):
    r = np.random.default_rng(5).uniform(lo, hi, n)
    r = np.round(r * 2.0 ** 20) / 2.0 ** 20
    assert np.all(r * r == (np.longdouble(r) * np.longdouble(r)).astype(float))
    return r


def lj_parts(r, n_rep):
    """Mie energies of the two atoms, and their larger parts, in extended precision."""
    n = np.float64(n_rep)
    sig = np.float64((3.166 + 2.9) * 0.5)
    cn = n / (n - 6.0) * np.power(n / 6.0, 6.0 / (n - 6.0))
    eps = np.longdouble(np.float64(cn * np.sqrt(np.float64(78.2 * 61.7))))
    x = np.longdouble(np.float64(sig * sig)) / (np.longdouble(r) * np.longdouble(r))
    rep, att = x ** (np.longdouble(n) / 2), x ** 3
    return eps * (rep - att), eps * np.maximum(rep, att)


def lj_bar(n_rep):
    return U * (max(1.1 * n_rep / 2 + 2.0, 12.0) + 5.3 + 2.0)


@pytest.mark.parametrize("n_rep", [12.0, 14.0, 15.3, 20.0, 28.4])
def test_trial_position_lj(n_rep):
    s = two_atoms(n_rep)
    b = Box(s)
    r = distances(4000)
    at = np.zeros((len(r), 3))
    at[:] = s.xyz[0]
    at[:, 0] += r
    en, _, _ = b.particle_inter(1, 0.0, at, skip_mol=1)
    e, scale = lj_parts(r, n_rep)
    assert np.max(np.abs((en - e) / scale)) <= lj_bar(n_rep)
    b.close()


@pytest.mark.parametrize("n_rep", [12.0, 15.3, 28.4])
def test_moved_molecule_lj(n_rep):
    """The change of a trial, from a place beyond the cutoff."""
    s = two_atoms(n_rep)
    s.xyz[1, 0] = 30.0
    b = Box(s)
    r = distances(400)
    e, scale = lj_parts(r, n_rep)
    new = s.xyz[0] + np.zeros((len(r), 1, 3))
    new[:, 0, 0] += r
    got = np.array([b.mol_inter(1, v)[0] for v in new])
    assert np.max(np.abs((got - e) / scale)) <= lj_bar(n_rep)
    b.close()


def second_atom_energies(n_rep, charge, r, call):
    s = two_atoms(n_rep, charge)
    b = Box(s)
    out = []
    for d in r:
        xyz = s.xyz.copy()
        xyz[1, 0] = xyz[0, 0] + d
        b.set_coords(xyz)
        out.append(call(b))
    b.close()
    return np.array(out).T


@pytest.mark.parametrize("n_rep,call", [(12.0, "box_inter"), (15.3, "box_inter"),
                                        (28.4, "box_inter"), (12.0, "box_force")])
def test_whole_box_lj(n_rep, call):
    r = distances(400)
    lj, _ = second_atom_energies(n_rep, 0.0, r, lambda b: getattr(b, call)()[:2])
    e, scale = lj_parts(r, n_rep)
    assert np.max(np.abs((lj - e) / scale)) <= lj_bar(n_rep)


def test_whole_box_coulomb_has_no_bias():
    m = ctypes.CDLL("libm.so.6")
    m.erfcl.restype, m.erfcl.argtypes = ctypes.c_longdouble, [ctypes.c_longdouble]
    r = distances(1600)
    _, real = second_atom_energies(12.0, 1.0, r, lambda b: b.box_inter())
    alpha = np.sqrt(-np.log(TOL)) / RC
    x = np.longdouble(alpha) * np.longdouble(r)
    hi = x.astype(float)
    erfc = np.array([m.erfcl(v) for v in hi])  # at the double nearest x, then moved to x
    slope = -2.0 / np.sqrt(np.pi) * np.exp(-hi * hi)
    e = -np.longdouble(167103.208067979) * (np.longdouble(erfc) + slope * (x - hi)) / r
    rel = ((real - e) / e).astype(float)
    assert np.sqrt(np.mean(rel * rel)) <= 1.6e-15
    assert abs(np.mean(rel)) <= 1.2e-16
