"""Mixed precision on disks whose one-sided items are narrowed (chunks halved,
one sink per lane): class sizes around the 64- and 128-sink items and the
256-source tile, against the FP64 oracle under the FP32 bound the other
mixed-precision tests hold every body to, and a batch of such disks against
the same disks alone, bit for bit."""
import numpy as np
import pytest

import oracle_lib as O
import redamd as R
from systems import small_system, as3, bits_equal

pytestmark = pytest.mark.gpu


def _disk(n_si, n_nsi, n_ni, seed, inactive=()):
    types = [0] + [3] * (n_si - 1) + [5] * n_nsi + [6] * n_ni
    return small_system(n_si + n_nsi + n_ni, seed, types, inactive=inactive)


def _mutual(r, v, p, b, nbt):
    """|a| without the star's pull (the part computed in FP32)."""
    q = p.copy()
    q["mass"][0] = 0.0
    rc, dy = O.ODisk(r, v, q, b, nbt).calc_dydx(1, 0, 0.0, r, v)
    assert rc == 0
    return np.linalg.norm(as3(dy), axis=1)


@pytest.mark.parametrize("pair_mode", [R.RD_PAIRS_SYMMETRIC, R.RD_PAIRS_ONE_SIDED])
@pytest.mark.parametrize("sinks", [1, 2, 4])
@pytest.mark.parametrize("sizes", [(2, 1, 1), (64, 64, 64), (65, 127, 129), (257, 255, 1), (1003, 1500, 498), (300, 2100, 700)])
def test_narrow_items(sizes, sinks, pair_mode):
    r, v, p, b, nbt = _disk(*sizes, seed=sum(sizes), inactive=(1, sizes[0], sum(sizes) - 1))
    d = R.Disk(r, v, p, b, nbt)
    d.set_precision(R.RD_PREC_MIXED)
    d.set_tuning(sinks_per_lane=sinks, pair_mode=pair_mode)
    a = as3(d.calc_dydx(1, 0, 0.0, r, v))
    rc, ody = O.ODisk(r, v, p, b, nbt).calc_dydx(1, 0, 0.0, r, v)
    assert rc == 0
    ref = as3(ody)
    err = np.linalg.norm(a - ref, axis=1)
    scale = _mutual(r, v, p, b, nbt)
    on = b["id"] > 0
    # FP32 pair terms of the mutual part; 1e-15 of the whole for its FP64 rest
    assert np.all(err[on] <= 2e-5 * scale[on] + 1e-15 * np.linalg.norm(ref, axis=1)[on])
    assert np.all(a[~on] == 0.0)


def test_batch_of_class_disks_matches_single_disks():
    parts = [_disk(*s, seed=70 + k) for k, s in enumerate([(300, 200, 40), (70, 3000, 10), (1200, 100, 900)])]
    cat = [np.concatenate([q[i] for q in parts]) for i in range(4)]
    bd = R.Disk(*cat, np.stack([q[4] for q in parts]), batch=True)
    bd.set_precision(R.RD_PREC_MIXED)
    for k, (r, v, p, b, nbt) in enumerate(parts):
        d = R.Disk(r, v, p, b, nbt)
        d.set_precision(R.RD_PREC_MIXED)
        assert bits_equal(d.calc_dydx(1, 0, 0.0, r, v), bd.calc_dydx(1, 0, 0.0, r, v, k=k))
