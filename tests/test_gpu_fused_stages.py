"""RKF7(8) stages and the operator done in the FP64 pair pass (items of 4 and 8
sinks) against the oracle, bit for bit: body counts around an item and around
the change of item size on a 256-CU device, rejected attempts (k0 kept), the
stage-0 pass run ahead of the next step (steps()) and not (step()), fixed
steps, error terms of test particles counted or not."""
import numpy as np
import pytest

import oracle_lib as O
import redamd as R
from systems import small_system, mixed_types, bits_equal

pytestmark = pytest.mark.gpu


def _pair(arrays, dt, adaptive=True, tol=1e-12):
    d, o = R.Disk(*arrays), O.ODisk(*arrays)
    return d, o, R.Integrator(d, R.RD_RKF78, dt, adaptive=adaptive, tol=tol), O.OInteg(o, 4, dt, adaptive=adaptive,
                                                                                   tol=tol)


def _same_state(d, o):
    _, rr, vv, _, _ = d.state()
    _, orr, ovv, _, _ = o.state()
    return bits_equal(rr, orr) and bits_equal(vv, ovv)


@pytest.mark.parametrize("ahead", [True, False])
@pytest.mark.parametrize("n", [2, 3, 5, 64, 257, 1024, 1025, 2048])
def test_rkf78_steps(n, ahead):
    # the first step is too long by far: attempts are rejected before one is accepted
    d, o, it, oi = _pair(R.make_disk(n - 1, 7 + n), 10.0 * R.K_GAUSS)
    if ahead:
        it.steps(3)
    else:
        for _ in range(3):
            it.step()
    for _ in range(3):
        oi.step()
    assert _same_state(d, o)


@pytest.mark.parametrize("n", [257, 1100])
def test_rkf78_fixed_steps(n):
    d, o, it, oi = _pair(R.make_disk(n - 1, 9), 0.1 * R.K_GAUSS, adaptive=False)
    it.steps(3)
    for _ in range(3):
        oi.step()
    assert _same_state(d, o)


@pytest.mark.parametrize("n", [90, 1300])
def test_rkf78_classes(n):
    """All classes, inactive bodies among them: only bodies before the test particles enter the error."""
    arrays = small_system(n, 60 + n, mixed_types(n), inactive=(5, n // 2, n - 1))
    arrays[2]["mass"][arrays[3]["body_type"] == R.BODY_TP] = 0.0
    d, o, it, oi = _pair(arrays, 1e-4, tol=1e-9)
    it.steps(2)
    for _ in range(2):
        oi.step()
    assert _same_state(d, o)


@pytest.mark.parametrize("k", [0, 1, 2])
def test_operator_in_a_batch(k):
    """Only the asked disk's records are written, whatever the others' sizes."""
    parts = [R.make_disk(n, 3 + n) for n in (5, 130, 62)]
    d = R.Disk(*[np.concatenate([q[i] for q in parts]) for i in range(4)], np.stack([q[4] for q in parts]),
               batch=True)
    r, v = parts[k][0], parts[k][1]
    dy = d.calc_dydx(1, 0, 0.0, r, v, k=k)
    rc, ody = O.ODisk(*parts[k]).calc_dydx(1, 0, 0.0, r, v)
    assert rc == 0 and bits_equal(dy, ody)
