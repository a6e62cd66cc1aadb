"""A box that the device move loop refuses while it prepares (more than 40
k-vectors along an axis) is refused again by the next call, and its host moves go
on.
"""
import pytest

from gomc_amd.api import Box, GomcError
from test_gpu_recip import water_in

pytestmark = pytest.mark.gpu


def test_refused_twice():
    b = Box(water_in((20.0, 20.0, 150.0), 60, 8.0))
    for _ in range(2):
        with pytest.raises(GomcError, match="more than 40 k-vectors per axis"):
            b.run(10, device=True)
    n, rec = b.run(10)
    assert len(rec["acc"]) == 10 and n == rec["acc"].sum()
    b.close()
