"""Mixed precision: the symmetric kernel's tiles cut into row and reaction items
(launches of few tiles) give the whole tiles' bits.  A disk alone is cut; in a
batch with a disk of many tiles it is not.  Sizes around rows, quarters and
blocks, the rule's limit, body classes, inactive bodies, a coincident pair."""
import numpy as np
import pytest

import redamd as R
from systems import small_system, mixed_types

pytestmark = pytest.mark.gpu

BIG = R.make_disk(7000, 17)   # 28 blocks: more tiles than the rule's limit


def _acc(parts, k=0):
    d = R.Disk(*[np.concatenate([q[i] for q in parts]) for i in range(4)], np.stack([q[4] for q in parts]),
               batch=True)
    d.set_precision(R.RD_PREC_MIXED)
    a = d.calc_dydx(1, 0, 0.0, parts[k][0], parts[k][1], k=k)
    return np.stack([a["x"], a["y"], a["z"]], 1).view(np.uint64)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129, 192, 193, 250, 256, 257, 448, 449, 513, 1000, 2047, 4095, 4097])
def test_split_matches_whole_tiles(n):
    r, v, p, b, nbt = small_system(n, 300 + n, inactive=tuple(range(3, n, 53)))
    if n > 2:
        for c in "xyz":
            r[c][n - 1] = r[c][1]
    part = (r, v, p, b, nbt)
    assert np.array_equal(_acc([part]), _acc([part, BIG]))


@pytest.mark.parametrize("n", [90, 700, 3001])
def test_split_with_one_sided_pairs(n):
    r, v, p, b, nbt = small_system(n, 400 + n, mixed_types(n), inactive=(5, n // 2, n - 1))
    p["mass"][b["body_type"] == R.BODY_TP] = 0.0
    part = (r, v, p, b, nbt)
    assert np.array_equal(_acc([part]), _acc([part, BIG]))
