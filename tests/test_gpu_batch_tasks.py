"""Task lists of a launch: more boxes than workgroups, of different and of no
moves.  A box's course does not depend on the boxes beside it, so each equals
the same box run alone to the last bit, whatever list it came to stand in."""
import numpy as np
import pytest

from gomc_amd import systems
from gomc_amd.api import Batch

pytestmark = pytest.mark.gpu

# one box, a few, as many as a device has workgroups and some more
@pytest.mark.parametrize("nboxes", [1, 7, 256, 290])
def test_every_box_runs_its_own_moves(nboxes):
    base = [systems.water_box(40 + 3 * (i % 4), rcut=5.0, tolerance=1e-5, seed=900 + i % 4) for i in range(nboxes)]
    counts = [[(5 * i + 3 * k) % 11 for i in range(nboxes)] for k in range(3)]
    bt = Batch(base)
    for c in counts:
        bt.run(np.array(c, dtype=np.int64))
    e, acc, done = bt.stats()
    assert done.tolist() == np.sum(counts, axis=0).tolist()
    times = bt.box_times()
    assert np.all(times[np.array(counts[-1]) > 0] > 0)
    for i in sorted({0, nboxes // 2, nboxes - 1, nboxes // 3}):
        one = Batch([base[i]])
        for c in counts:
            one.run(np.array([c[i]], dtype=np.int64))
        e1, acc1, done1 = one.stats()
        assert np.array_equal(e1[0], e[i]) and acc1[0] == acc[i] and done1[0] == done[i]
        for p, q in zip(one.coords(0), bt.coords(i)):
            assert np.array_equal(p, q)
        one.close()
    bt.close()
