"""Passes of two moves in the batched kernel: an even step and the odd step
after it share a pass, the odd one's energies found for both outcomes of the
even one.  The cases where the pairing breaks or matters most: few molecules
(both draws pick the same one, or near ones), the move settings adjusted every
few steps, launches that end between the two steps, rigid kinds of one and
three atoms, teams, and no Ewald.

Bar: the oracle's decisions move for move and energies to 1e-10 of their
scale, as for every batched box; a run cut at odd steps equals the same run in
one launch bit for bit (a move's sums have the same terms in the same order
whether or not it shares its pass).
"""
import numpy as np
import pytest

from gomc_amd import systems
from gomc_amd.api import Batch
from oracle.pyoracle import Oracle

pytestmark = pytest.mark.gpu


def methane_box(n, seed):
    kinds = [systems.methane_kind(0)]
    mk = np.zeros(n, np.int32)
    box = (n / 0.008) ** (1.0 / 3.0)
    xyz = systems.place_molecules(kinds, mk, box, seed, min_heavy=3.2, min_any=3.2)
    return systems.System(box=(box,) * 3, temperature=200.0, rcut=min(10.0, box / 2), rcut_low=1.0,
                          rcut_coulomb=min(10.0, box / 2), tolerance=1e-5, kinds=kinds, mol_kind=mk,
                          xyz=xyz, seed=seed, ewald=False, electrostatic=False, sigma=[3.73],
                          epsilon=[148.0], n_rep=[12.0])


CASES = {
    "ten_waters": (lambda: systems.water_box(10, density=0.1, seed=5, adj_steps=100), 3000, None),
    "adjust_every_3": (lambda: systems.water_box(60, density=0.5, seed=6, adj_steps=3), 1501, None),
    "adjust_every_step": (lambda: systems.water_box(40, density=0.5, seed=7, adj_steps=1), 400, None),
    "methane": (lambda: methane_box(120, 8), 3000, None),
    "no_cull_200": (lambda: systems.water_box(200, seed=9), 1200, None),
    "cull_900": (lambda: systems.water_box(900, seed=10), 1201, None),
    "team4_900": (lambda: systems.water_box(900, seed=11, adj_steps=500), 1200,
                  {"team_min": [0, 400, 0]}),
    "team8_500": (lambda: systems.water_box(500, seed=12), 901, {"team_min": [0, 0, 300]}),
}


@pytest.mark.parametrize("name", CASES)
def test_oracle_sequence(name):
    make, n, tuning = CASES[name]
    s = make()
    o = Oracle(s, threads=8)
    e0 = np.abs(o.energies())
    bt = Batch([s], tuning=tuning or "default")
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
@pytest.mark.parametrize("name", ["ten_waters", "methane", "no_cull_200", "cull_900", "team4_900"])
def test_cut_at_odd_steps_same_bits(name, precision):
    make, _, tuning = CASES[name]
    n = 600
    one = Batch([make()], precision=precision, tuning=tuning or "default")
    one.run([n])
    cut = Batch([make()], precision=precision, tuning=tuning or "default")
    left = n
    for k in (1, 2, 7, 65, 64, 129, 3):
        cut.run([k])
        left -= k
    cut.run([left])
    assert np.array_equal(one.stats()[0], cut.stats()[0])
    assert np.array_equal(one.stats()[1], cut.stats()[1])
    assert np.array_equal(one.coords(0), cut.coords(0))
    one.close()
    cut.close()
