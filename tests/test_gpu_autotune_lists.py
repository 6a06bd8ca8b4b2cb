"""rd_autotune on a disk whose one-sided items are narrowed: the settings that make
the same launch are timed once, so the first of them is chosen, not one by
timing noise; and the launch of narrow items is the one-sink-per-lane kernel
whatever the limit, with the same bits."""
import numpy as np
import pytest

import redamd as R
from systems import small_system, bits_equal

pytestmark = pytest.mark.gpu


def _disk():
    types = [0] + [3] * 299 + [5] * 200 + [6] * 100
    return small_system(600, 77, types)


def test_autotune_times_a_launch_once():
    r, v, p, b, nbt = _disk()
    d = R.Disk(r, v, p, b, nbt)
    d.set_precision(R.RD_PREC_MIXED)
    best = d.autotune()
    assert (best.sinks_per_lane, best.chunk, best.blocks_per_cu) == (1, 512, 1)


def test_narrow_items_do_not_depend_on_the_limit():
    r, v, p, b, nbt = _disk()
    out = []
    for sinks in (1, 2, 4):
        d = R.Disk(r, v, p, b, nbt)
        d.set_precision(R.RD_PREC_MIXED)
        d.set_tuning(sinks_per_lane=sinks)
        out.append(d.calc_dydx(1, 0, 0.0, r, v))
    assert bits_equal(out[0], out[1]) and bits_equal(out[0], out[2])
