"""Snapshots around the staging buffer's size (8192 bodies a slice): the records
come back as they went in, alone and from a disk inside a batch."""
import numpy as np
import pytest

import redamd as R
from systems import small_system, bits_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 8191, 8192, 8193, 16384, 24577])
def test_state_returns_the_records(n):
    parts = [small_system(5, 1), small_system(n, 2)]
    for one in ([parts[1]], parts):
        d = R.Disk(*[np.concatenate([q[i] for q in one]) for i in range(4)], np.stack([q[4] for q in one]),
                   batch=True)
        for k, q in enumerate(one):
            t, r, v, p, b = d.state(k)
            assert t == 0.0 and all(bits_equal(a, w) for a, w in zip((r, v, p, b), q))
