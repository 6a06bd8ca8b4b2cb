"""A disk whose bodies were all removed (every body ejected, then
rd_rebuild_vectors): calls on it do nothing, and the other disks of its batch
are untouched."""
import numpy as np
import pytest

import oracle_lib as O
import redamd as R
from systems import small_system, bits_equal
from test_gpu_device_dydx import DevArray

pytestmark = pytest.mark.gpu

THR = (0.0, 50.0, 0.0)   # ejection beyond 50 AU


def _far(n, seed):
    """n protoplanets without a star, all past the ejection distance."""
    r, v, p, b, nbt = small_system(n, seed, [3] * n)
    r["x"] += 100.0
    return r, v, p, b, nbt


def _eject_all(d, k):
    d.check_ejection_hit_centrum(k)
    d.handle_ejection_hit_centrum(k)
    d.clear_event_counter(k)
    d.rebuild_vectors(k)
    assert d.n_total(k) == 0


@pytest.mark.parametrize("k", [0, 1, 2])
@pytest.mark.parametrize("prec", [R.RD_PREC_FP64, R.RD_PREC_MIXED])
def test_operator_on_an_empty_disk_of_a_batch(prec, k):
    parts = [R.make_disk(n, 3 + n) for n in (60, 130)]
    parts.insert(k, _far(3, 8))
    d = R.Disk(*[np.concatenate([q[i] for q in parts]) for i in range(4)], np.stack([q[4] for q in parts]),
               threshold=THR, batch=True)
    d.set_precision(prec)
    _eject_all(d, k)
    # leaves the control flags of every disk set, as a run of fixed steps does
    R.Integrator(d, R.RD_RK4, 1e-3, adaptive=False).steps(1)
    before = [d.state(q)[1:3] for q in range(3)]
    none = np.zeros(0, R.VAR4)
    assert len(d.calc_dydx(1, 0, 0.0, none, none, k=k)) == 0
    guard = np.full(4 * 300, 7.0).view(R.VAR4)
    bufs = [DevArray(guard.nbytes) for _ in range(3)]
    for q in bufs:
        q.put(guard)
    d.calc_dydx_device(1, 0, 0.0, *[q.p.value for q in bufs], k=k)
    for q in bufs:
        assert bits_equal(q.get(np.zeros(300, R.VAR4)), guard)
    for q in range(3):
        assert all(bits_equal(a, w) for a, w in zip(d.state(q)[1:3], before[q]))
    if prec == R.RD_PREC_FP64:
        for q in range(3):
            if q == k:
                continue
            rr, vv = before[q]
            rc, ody = O.ODisk(*parts[q]).calc_dydx(1, 0, 0.0, rr, vv)
            assert rc == 0 and bits_equal(d.calc_dydx(1, 0, 0.0, rr, vv, k=q), ody)


@pytest.mark.parametrize("steps", [False, True])
@pytest.mark.parametrize("method", [R.RD_RKF78, R.RD_RK4])
def test_adaptive_steps_of_an_empty_disk(method, steps):
    """No body, no error: every attempt is accepted and the step doubles (the
    reference's rule for an error of zero)."""
    d = R.Disk(*_far(3, 8), threshold=THR)
    _eject_all(d, 0)
    it = R.Integrator(d, method, 1e-3, adaptive=True, tol=1e-10)
    it.set_guard(max_attempts=4)
    if steps:
        it.steps(2)
    else:
        assert it.step() == 1e-3 and it.step() == 2e-3
    assert it.dt_next() == 4e-3
