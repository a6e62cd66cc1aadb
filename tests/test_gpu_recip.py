"""Whole-box reciprocal space (structure factors, k-space forces, the
virial's reciprocal term) against the oracle at the sizes where the matrix
products can go wrong: boxes of unequal edges, fewer columns than one unit,
more than one window of nz (long in z), no room for the x and y tables (long
in x), atom counts around the tiles, and uncharged and reservoir atoms.

Bar: sums and forces within 1e-12 of their largest value.  A phase is at most
7 complex products from a sincos whose argument is n r / L to one rounding:
about 2 pi n 1.1e-16 + 7 x 2.2e-16, 2e-15 at n = 40 and 2e-12 at n = 2400.
"""
import numpy as np
import pytest

from gomc_amd import systems
from gomc_amd.api import Box
from oracle.pyoracle import Oracle

pytestmark = pytest.mark.gpu


def water_in(box, n, rcut, seed=3):
    """n waters in a box of the given edges, on a jittered grid."""
    rng = np.random.default_rng(seed)
    box = np.asarray(box, float)
    div = np.maximum(1, np.floor(box / 4.5)).astype(int)
    grid = np.stack(np.meshgrid(*(np.arange(d) for d in div), indexing="ij"), -1).reshape(-1, 3)
    cell = grid[rng.permutation(len(grid))[:n]]
    assert len(cell) == n
    geo = systems.water_kind().geometry
    xyz = []
    for c in cell:
        q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
        xyz.append((c + 0.5 + rng.uniform(-0.1, 0.1, 3)) * box / div + geo @ q.T)
    xyz = np.mod(np.concatenate(xyz), box)
    return systems.System(box=tuple(box), temperature=300.0, rcut=rcut, rcut_low=1.0,
                          rcut_coulomb=rcut, tolerance=1e-5, kinds=[systems.water_kind()],
                          mol_kind=np.zeros(n, np.int32), xyz=xyz, seed=seed,
                          **systems.WATER_TYPES)


def check_sums(b, o, tol):
    g, (re, im) = b.recip_get(), o.recip_sums()
    top = max(np.abs(re).max(), np.abs(im).max())
    assert np.abs(g["sum_r"] - re).max() <= tol * top
    assert np.abs(g["sum_i"] - im).max() <= tol * top


CASES = [((18.1, 18.1, 18.1), 1, 9.0), ((18.1, 18.1, 18.1), 21, 9.0), ((19.0, 31.0, 24.0), 86, 9.0),
         ((20.0, 20.0, 150.0), 171, 8.0), ((20.0, 95.0, 20.0), 128, 9.5),
         ((6000.0, 18.5, 18.5), 40, 9.0)]


@pytest.mark.parametrize("box,n,rcut", CASES)
def test_sums_forces_virial(box, n, rcut):
    s = water_in(box, n, rcut)
    b, o = Box(s), Oracle(s, threads=8)
    tol = 1e-12 if max(box) < 1000 else 1e-11
    t, ot = b.system_total(), o.system_total()
    assert np.allclose(t, ot, rtol=10 * tol, atol=0)
    check_sums(b, o, tol)
    fa, fm = b.box_force_recip()
    oa, om = o.box_force_recip()
    assert np.abs(fa - oa).max() <= 10 * tol * np.abs(oa).max()
    assert np.abs(fm - om).max() <= 10 * tol * np.abs(oa).max()
    v, ov = b.virial(), o.virial()
    assert abs(v["recip"] - ov["recip"]) <= 100 * tol * abs(ov["recip"])
    b.close()
    o.close()


def test_uncharged_and_reservoir_atoms_add_nothing():
    s = systems.gcmc_mixture(30, 21, 24.0, reservoir=40, seed=5)
    b, o = Box(s), Oracle(s, threads=8)
    check_sums(b, o, 1e-12)
    b.close()
    o.close()
