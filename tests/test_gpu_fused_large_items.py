"""RKF7(8) and RK4 stages done in the FP64 pair pass on items of 12 and 18 sinks,
against the oracle, bit for bit: body counts on both sides of the changes of item
size and of the number of blocks a CU (256-CU device), rejected attempts, the
stage-0 pass run ahead of the next step and not, fixed steps, all classes with
inactive bodies and the error terms that count."""
import numpy as np
import pytest

import oracle_lib as O
import redamd as R
from systems import small_system, mixed_types, bits_equal

pytestmark = pytest.mark.gpu


def _run(arrays, method, dt, steps, adaptive=True, tol=1e-12, ahead=True, tp=0):
    d, o = R.Disk(*arrays), O.ODisk(*arrays)
    it = R.Integrator(d, method, dt, adaptive=adaptive, tol=tol)
    oi = O.OInteg(o, method, dt, adaptive=adaptive, tol=tol)
    if tp:
        it.set_error_check_for_tp(True)
        O.lib.or_set_error_check_for_tp(oi.h, 1)
    if ahead:
        it.steps(steps)
    else:
        for _ in range(steps):
            it.step()
    for _ in range(steps):
        oi.step()
    _, rr, vv, _, _ = d.state()
    _, orr, ovv, _, _ = o.state()
    assert bits_equal(rr, orr) and bits_equal(vv, ovv)
    assert it.dt_next() == oi.dt_next()


# 12 sinks, one block a CU; 18, one; 12, two; and the separate kernels beyond
@pytest.mark.parametrize("n", [2049, 3072, 3073, 4608, 4609])
def test_rkf78(n):
    _run(R.make_disk(n - 1, 7 + n), R.RD_RKF78, 5.0 * R.K_GAUSS, 2, ahead=n % 2 == 0)


@pytest.mark.parametrize("n", [2049, 3072, 3073, 4608, 4609, 6144, 6145])
def test_rk4_fixed(n):
    _run(R.make_disk(n - 1, 9 + n), R.RD_RK4, 0.1 * R.K_GAUSS, 2, adaptive=False)


@pytest.mark.parametrize("n", [2500, 4000])
def test_rkf78_fixed(n):
    _run(R.make_disk(n - 1, 9), R.RD_RKF78, 0.1 * R.K_GAUSS, 2, adaptive=False)


@pytest.mark.parametrize("tp", [0, 1])
@pytest.mark.parametrize("n", [2600, 4200])
def test_rkf78_classes(n, tp):
    arrays = small_system(n, 60 + n, mixed_types(n), inactive=(5, n // 2, n - 1))
    arrays[2]["mass"][arrays[3]["body_type"] == R.BODY_TP] = 0.0
    _run(arrays, R.RD_RKF78, 1e-4, 1, tol=1e-9, tp=tp)
