"""Mixed precision on disks whose one-sided items stay wide: 128 and 256 sinks
each (2 and 4 per lane) in their own kernel, beside whole symmetric tiles and
beside tiles cut finer, and a class of few sinks and so many sources that its
chunks stay whole; ragged last groups and chunks, inactive bodies.  Against the
FP64 oracle under the bound the other mixed-precision tests use.  Item counts
in the ids' comments are for a 256-CU device (the rule asks for 512)."""
import numpy as np
import pytest

import oracle_lib as O
import redamd as R
from systems import as3, small_system

pytestmark = pytest.mark.gpu


def _disk(n_si, n_nsi, n_ni, seed):
    n = n_si + n_nsi + n_ni
    types = [0] + [3] * (n_si - 1) + [5] * n_nsi + [6] * n_ni
    return small_system(n, seed, types, inactive=tuple({1, min(n_si, n - 2), n - 1}))


def _mutual(r, v, p, b, nbt):
    q = p.copy()
    q["mass"][0] = 0.0
    rc, dy = O.ODisk(r, v, q, b, nbt).calc_dydx(1, 0, 0.0, r, v)
    assert rc == 0
    return np.linalg.norm(as3(dy), axis=1)


@pytest.mark.parametrize("sizes,sinks,pair_mode", [
    ((6003, 0, 0), 4, R.RD_PAIRS_ONE_SIDED),        # 24 groups of 256 x 24 chunks, no symmetric items
    ((3005, 4500, 1503), 2, R.RD_PAIRS_SYMMETRIC),  # beside 78 whole tiles
    ((3005, 4500, 1503), 4, R.RD_PAIRS_SYMMETRIC),
    ((31, 60100, 0), 2, R.RD_PAIRS_SYMMETRIC),      # beside cut tiles: few SI bodies, many NSI ones
    ((31, 120100, 0), 4, R.RD_PAIRS_SYMMETRIC),
    ((1, 40001, 0), 2, R.RD_PAIRS_SYMMETRIC),       # the star's sources keep their chunk
])
def test_wide_items(sizes, sinks, pair_mode):
    r, v, p, b, nbt = _disk(*sizes, seed=sum(sizes))
    d = R.Disk(r, v, p, b, nbt)
    d.set_precision(R.RD_PREC_MIXED)
    d.set_tuning(sinks_per_lane=sinks, pair_mode=pair_mode)
    a = as3(d.calc_dydx(1, 0, 0.0, r, v))
    rc, ody = O.ODisk(r, v, p, b, nbt).calc_dydx(1, 0, 0.0, r, v)
    assert rc == 0
    ref = as3(ody)
    err = np.linalg.norm(a - ref, axis=1)
    on = b["id"] > 0
    # FP32 pair terms of the mutual part; 1e-15 of the whole for its FP64 rest
    assert np.all(err[on] <= 2e-5 * _mutual(r, v, p, b, nbt)[on] + 1e-15 * np.linalg.norm(ref, axis=1)[on])
    assert np.all(a[~on] == 0.0)
