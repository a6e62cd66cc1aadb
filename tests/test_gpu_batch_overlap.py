"""The batched kernel's overlap test where RcutLow exceeds the cutoff: only a
pair inside the cutoff is one, however large RcutLow, with the centre cull and
without.  Dilute boxes, so that a moved molecule often has neighbours between
the two radii and none inside the cutoff.

Bar: the oracle's decisions and overlaps move for move.
"""
import numpy as np
import pytest

from gomc_amd import systems
from gomc_amd.api import Batch
from oracle.pyoracle import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n,box,cull", [(40, 45.0, True), (4, 22.0, False)])
def test_overlap_needs_the_cutoff(n, box, cull, precision):
    s = systems.water_box(n, box=box, seed=21)
    s.rcut_low = 14.0
    moves = 400
    bt = Batch([s], precision=precision, tuning="default")
    assert bt.layout(0)["cull"] == cull
    bt.set_trace(0, moves)
    bt.run([moves])
    tr = bt.trace()
    o = Oracle(s, threads=4)
    _, ro = o.run(moves, mode=1)
    assert 0 < ro["acc"].sum() < moves
    assert np.array_equal(tr["acc"], ro["acc"])
    bt.close()
    o.close()
