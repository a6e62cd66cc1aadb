"""The batched kernel on rigid kinds of two and four atoms (four fill the wave
that takes the cross terms of a pass's two moves), with and without the centre
cull, on one workgroup and on teams, and on cutoffs beyond 16 A, against the
oracle move for move.

Bar: that of the other batched boxes: the oracle's decisions, energy changes to
1e-10 of their scale, coordinates to 1e-9 A.  A box's run does not depend on how
launches cut it: bit for bit.
"""
import numpy as np
import pytest

from gomc_amd import systems
from gomc_amd.api import Batch
from oracle.pyoracle import Oracle
from rigid_chains import chain_box, chain_kind

pytestmark = pytest.mark.gpu


def chains(atoms, n, edge, **kw):
    return chain_box([chain_kind(atoms, 2)], [0] * n, (edge,) * 3, 2, **kw)


CASES = {
    "2_atoms_no_cull": (lambda: chains(2, 100, 17.0), 900, None, False),
    "2_atoms_cull": (lambda: chains(2, 600, 34.0), 700, None, True),
    "4_atoms_few": (lambda: chains(4, 6, 20.0), 1500, None, False),
    "4_atoms_no_cull": (lambda: chains(4, 90, 20.0), 700, None, False),
    "4_atoms_cull": (lambda: chains(4, 400, 36.0), 500, None, True),
    "4_atoms_team": (lambda: chains(4, 400, 36.0, seed=5), 500, {"team_min": [0, 300, 0]}, True),
    "2_atoms_no_ewald": (lambda: chains(2, 150, 24.0, ewald=False), 700, None, True),
    "rcut_18": (lambda: systems.water_box(1700, rcut=18.0, seed=4), 150, None, False),
    "rcut_5": (lambda: systems.water_box(400, rcut=5.0, seed=4), 500, None, True),
}


@pytest.mark.parametrize("name", CASES)
def test_oracle_sequence(name):
    make, n, tuning, cull = CASES[name]
    s = make()
    o = Oracle(s, threads=8)
    e0 = np.abs(o.energies())
    bt = Batch([s], tuning=tuning or "default")
    assert bt.layout(0)["cull"] == cull
    bt.set_trace(0, n)
    bt.run([n])
    tr = bt.trace()
    no, ro = o.run(n, mode=1)
    assert np.array_equal(tr["acc"], ro["acc"]), np.nonzero(tr["acc"] != ro["acc"])[0][:5]
    for k, i in (("dlj", 0), ("dreal", 2), ("drecip", 3)):
        live = ro["ovl"] == 0
        err = np.abs(tr[k] - ro[k])[live]
        assert np.all(err <= 1e-10 * np.maximum(np.abs(ro[k])[live], max(e0[i], 1.0))), k
    e, acc, done = bt.stats()
    assert done[0] == n and acc[0] == no
    assert np.allclose(bt.coords(0), o.coords(), rtol=0, atol=1e-9)
    bt.close()
    o.close()


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("name", ["2_atoms_cull", "4_atoms_few", "4_atoms_no_cull", "4_atoms_team"])
def test_cut_launches_same_bits(name, precision):
    make, _, tuning, _ = CASES[name]
    n = 300
    one = Batch([make()], precision=precision, tuning=tuning or "default")
    one.run([n])
    cut = Batch([make()], precision=precision, tuning=tuning or "default")
    left = n
    for k in (1, 2, 7, 64, 65):
        cut.run([k])
        left -= k
    cut.run([left])
    assert np.array_equal(one.stats()[0], cut.stats()[0])
    assert np.array_equal(one.stats()[1], cut.stats()[1])
    assert np.array_equal(one.coords(0), cut.coords(0))
    one.close()
    cut.close()


def test_boxes_of_several_tables():
    """Boxes of different alpha and cutoff in one batch, two sharing each table:
    every box equals the same box alone."""
    def make():
        out = []
        for i, (rc, tol) in enumerate(((9.0, 1e-5), (10.0, 1e-6), (9.0, 1e-5), (17.0, 1e-5), (10.0, 1e-6))):
            out.append(systems.water_box(1500 if rc > 10 else 300, rcut=rc, tolerance=tol, seed=30 + i))
        return out
    both = Batch(make(), tuning="default")
    both.run([40] * 5)
    e = both.stats()[0]
    for i, s in enumerate(make()):
        alone = Batch([s], tuning="default")
        alone.run([40])
        assert np.array_equal(alone.stats()[0][0], e[i])
        assert np.array_equal(alone.coords(0), both.coords(i))
        alone.close()
    both.close()
