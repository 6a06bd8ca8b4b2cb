"""The FP64 pair kernel's items for few sources (batches of small disks, and the
pair pass of a small disk in gas) against the oracle, bit for bit: body counts
around its 4- and 16-sink items and 32- and 64-source tiles, the largest it
takes and one more, inactive bodies without a position, masses outside the
short root and division sequences."""
import numpy as np
import pytest

import oracle_lib as O
import redamd as R
from systems import small_system, bits_equal

pytestmark = pytest.mark.gpu


def _batch(parts):
    return R.Disk(*[np.concatenate([q[i] for q in parts]) for i in range(4)], np.stack([q[4] for q in parts]),
                  batch=True)


def _oracle_step(part, h):
    o = O.ODisk(*part)
    O.OInteg(o, 2, h, adaptive=False).step()
    return o.state()[1:3]


# 20 disks: 4-sink items; 600: 16-sink items, 2048 blocks and more
@pytest.mark.parametrize("n_disk,sizes", [(20, (1, 2, 4, 5, 31, 33, 63, 64, 65, 130)), (20, (224, 16, 17)),
                                          (20, (225, 3)), (600, (2, 15, 16, 17, 32, 33, 64)), (60, (224, 97, 129))])
def test_batches_of_small_disks(n_disk, sizes):
    parts = []
    for k in range(n_disk):
        n = sizes[k % len(sizes)]
        part = small_system(n, 3000 + k, inactive=(n - 1,) if n > 4 else ())
        r, v, p, b, nbt = part
        if n > 4:
            r["x"][n - 1] = (np.nan, np.inf)[k % 2]
        if n > 20:
            p["mass"][[7, 8, 9]] = 1e-95, 1e95 if k % 5 == 0 else 0.0, -1e-9
        parts.append(part)
    d = _batch(parts)
    h = 1e-3
    before = [d.calc_dydx(1, 0, 0.0, q[0], q[1], k=k) for k, q in enumerate(parts[:8])]
    for q, dy in zip(parts, before):
        rc, ody = O.ODisk(*q).calc_dydx(1, 0, 0.0, q[0], q[1])
        on = q[3]["id"] > 0
        assert rc == 0 and bits_equal(dy[on], ody[on])
    R.Integrator(d, R.RD_RK4, h, adaptive=False).steps(1)
    for k in list(range(0, n_disk, max(1, n_disk // 40))) + [n_disk - 1]:
        _, rr, vv, _, _ = d.state(k)
        orr, ovv = _oracle_step(parts[k], h)
        on = parts[k][3]["id"] > 0
        assert bits_equal(rr[on], orr[on]) and bits_equal(vv[on], ovv[on]), k


@pytest.mark.parametrize("n", [2, 5, 33, 63, 64, 65])
def test_pair_pass_of_a_small_disk_in_gas(n):
    """Stages of a disk in gas are launches of their own; the drag acts on planetesimals only,
    of which there are none, so the steps are the oracle's bit for bit."""
    part = small_system(n, 77 + n)
    d = R.Disk(*part, gas=R.gas_params())
    h = 1e-3
    R.Integrator(d, R.RD_RK4, h, adaptive=False).steps(2)
    o = O.ODisk(*part)
    oi = O.OInteg(o, 2, h, adaptive=False)
    oi.step()
    oi.step()
    assert all(bits_equal(a, w) for a, w in zip(d.state()[1:3], o.state()[1:3]))
