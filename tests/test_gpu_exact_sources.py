"""The FP64 pair kernels' sources outside the ordinary: inactive ones whose
position is not finite (skipped, as the reference skips them) and single masses
outside the short root and division sequences, in the kernel with one sink per
lane and in every term-parallel item shape, against the oracle bit for bit."""
import numpy as np
import pytest

import oracle_lib as O
import redamd as R
from systems import small_system, bits_equal

pytestmark = pytest.mark.gpu


def _check(parts, ks):
    d = R.Disk(*[np.concatenate([q[i] for q in parts]) for i in range(4)], np.stack([q[4] for q in parts]),
               batch=True)
    for k in ks:
        r, v = parts[k][0], parts[k][1]
        rc, ody = O.ODisk(*parts[k]).calc_dydx(1, 0, 0.0, r, v)
        assert rc == 0
        dy = d.calc_dydx(1, 0, 0.0, r, v, k=k)
        on = parts[k][3]["id"] > 0
        assert np.all(np.isfinite(ody["x"][on])) and bits_equal(dy[on], ody[on]), k


def _lost(part, bodies):
    r, v, p, b, nbt = part
    for i, x in zip(bodies, (np.nan, np.inf, -np.inf)):
        b["id"][i] = -abs(b["id"][i])
        r["x"][i] = r["y"][i] = r["z"][i] = x
    return r, v, p, b, nbt


# 4, 8, 12 and 18 sinks per item on a 256-CU device; the last source is the one
# that padding repeats
@pytest.mark.parametrize("n", [90, 1300, 2600, 5000])
def test_inactive_sources_without_a_position(n):
    _check([_lost(small_system(n, 90 + n), (7, n // 2, n - 1))], [0])


def test_inactive_sources_without_a_position_lane():
    # at least 1024 groups of 256 sinks: one sink per lane
    parts = [small_system(1025, 700 + k) for k in range(260)]
    parts[3] = _lost(parts[3], (1, 600, 1024))
    _check(parts, [2, 3, 259])


@pytest.mark.parametrize("mass", [1e-95, 1e95, 5e-324])
def test_one_mass_outside_the_short_sequences_lane(mass):
    parts = [small_system(1025, 700 + k) for k in range(260)]
    parts[3][2]["mass"][500] = mass
    _check(parts, [2, 3])
