"""FP64 paths that no other test reaches: a launch of more items than blocks, in
which every block works through several items with the roles it took at its
start, and the operator on device arrays against the oracle (the host entry
point goes through the same kernels)."""
import numpy as np
import pytest

import oracle_lib as O
import redamd as R
from systems import small_system, mixed_types, as3, bits_equal
from test_gpu_device_dydx import DevArray

pytestmark = pytest.mark.gpu


# 7500 items of 18 sinks and 3000 of 16 (8 blocks a CU: 2048 on 256 CUs), fewer than
# the 1024 groups of 256 that take one sink per lane
@pytest.mark.parametrize("n_disk,n", [(500, 257), (600, 65)])
def test_blocks_of_several_items(n_disk, n):
    """One fixed RK4 step advances all disks, so every item of every launch works."""
    parts = [R.make_disk(n - 1, 1200 + k) for k in range(n_disk)]
    d = R.Disk(*[np.concatenate([q[i] for q in parts]) for i in range(4)], np.stack([q[4] for q in parts]),
               batch=True)
    h = 0.1 * R.K_GAUSS
    R.Integrator(d, R.RD_RK4, h, adaptive=False).steps(1)
    for k in list(range(0, n_disk, 37)) + [n_disk - 2, n_disk - 1]:
        o = O.ODisk(*parts[k])
        O.OInteg(o, 2, h, adaptive=False).step()
        _, rr, vv, _, _ = d.state(k)
        _, orr, ovv, _, _ = o.state()
        assert bits_equal(rr, orr) and bits_equal(vv, ovv), k


# operator in the pair pass (items of 4 sinks, with gas and without, and of 8) and after it
@pytest.mark.parametrize("n,gas", [(700, False), (700, True), (1500, False), (1500, True), (3000, False)])
def test_device_dydx_equals_the_oracle(n, gas):
    r, v, p, b, nbt = small_system(n, 51, mixed_types(n), inactive=(5, 300))
    g = R.gas_params() if gas else None
    d = R.Disk(r, v, p, b, nbt, t=2.0, gas=g)
    r2, v2 = r.copy(), v.copy()
    r2["x"] += 1e-3
    v2["y"] *= 0.99
    bufs = [DevArray(r.nbytes) for _ in range(3)]
    bufs[0].put(np.ascontiguousarray(r2))
    bufs[1].put(np.ascontiguousarray(v2))
    d.calc_dydx_device(1, 3, 2.5, *[q.p.value for q in bufs])
    got = bufs[2].get(np.zeros(n, R.VAR4))
    rc, want = O.ODisk(r, v, p, b, nbt, t=2.0, gas=g).calc_dydx(1, 3, 2.5, r2, v2)
    assert rc == 0
    if gas:   # device pow and exp in the drag
        ref = as3(want)
        assert np.all(np.abs(as3(got) - ref) <= 1e-13 * np.abs(ref).max(axis=1, keepdims=True))
    else:
        assert bits_equal(got, want)
