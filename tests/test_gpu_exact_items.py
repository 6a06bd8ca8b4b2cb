"""The FP64 pair kernel's item shapes (4, 8, 12 and 18 sinks) against the
oracle, bit for bit: body counts on both sides of each shape's limit on a
256-CU device, source counts around the 32- and 128-source tiles, classes with
partial items, inactive bodies, and masses outside the short root and division
sequences (every pair then takes the library's)."""
import numpy as np
import pytest

import oracle_lib as O
import redamd as R
from systems import small_system, mixed_types, bits_equal

pytestmark = pytest.mark.gpu


def _forces(r, v, p, b, nbt):
    d = R.Disk(r, v, p, b, nbt)
    o = O.ODisk(r, v, p, b, nbt)
    dy = d.calc_dydx(1, 0, 0.0, r, v)
    rc, ody = o.calc_dydx(1, 0, 0.0, r, v)
    assert rc == 0
    return dy, ody


@pytest.mark.parametrize("n", [3, 4, 5, 31, 33, 127, 128, 129, 1024, 1025, 2048, 2049, 3072, 3073, 4608, 4609, 6001])
def test_item_shapes(n):
    r, v, p, b, nbt = small_system(n, 40 + n, inactive=tuple(range(2, n, 97)))
    dy, ody = _forces(r, v, p, b, nbt)
    assert bits_equal(dy, ody)


@pytest.mark.parametrize("n", [90, 1300, 2600, 5000])
def test_item_shapes_classes(n):
    r, v, p, b, nbt = small_system(n, 60 + n, mixed_types(n), inactive=(5, n // 2, n - 1))
    p["mass"][b["body_type"] == R.BODY_TP] = 0.0
    dy, ody = _forces(r, v, p, b, nbt)
    assert bits_equal(dy, ody)


@pytest.mark.parametrize("mass", [1e-95, 1e95, 5e-324])
@pytest.mark.parametrize("n", [200, 1500, 2500, 5000])
def test_masses_outside_the_short_sequences(n, mass):
    r, v, p, b, nbt = small_system(n, 80 + n)
    p["mass"][n // 3] = mass
    p["mass"][n // 4] = 0.0
    p["mass"][n // 5] = -1e-9     # pulls (pushes) like any other
    dy, ody = _forces(r, v, p, b, nbt)
    assert bits_equal(dy, ody)


@pytest.mark.parametrize("n", [1023, 1025, 2047])
def test_rk4_fixed_steps(n):
    """4- and 8-sink items with the RK4 stage in the pair pass."""
    r, v, p, b, nbt = R.make_disk(n - 1, 5)
    d = R.Disk(r, v, p, b, nbt)
    o = O.ODisk(r, v, p, b, nbt)
    h = 0.1 * R.K_GAUSS
    it = R.Integrator(d, R.RD_RK4, h, adaptive=False)
    oi = O.OInteg(o, 2, h, adaptive=False)
    it.steps(3)
    for _ in range(3):
        oi.step()
    _, rr, vv, _, _ = d.state()
    _, orr, ovv, _, _ = o.state()
    assert bits_equal(rr, orr) and bits_equal(vv, ovv)
