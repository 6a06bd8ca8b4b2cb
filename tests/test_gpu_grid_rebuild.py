"""The gas grid outlives rd_rebuild_vectors, which lays every other buffer out
anew: the drag after a rebuild is that of a new disk of the bodies left, with
the same grid."""
import numpy as np
import pytest

import redamd as R
from systems import small_system, mixed_types, bits_equal, fargo_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [R.RD_PREC_FP64, R.RD_PREC_MIXED])
def test_grid_drag_after_a_rebuild(prec):
    n = 300
    r, v, p, b, nbt = small_system(n, 19, mixed_types(n))
    gone = [40, 150, 260]
    r["x"][gone] += 100.0     # past the ejection distance
    grid = fargo_grid(20, 64, 5, rho1=30.0)
    d = R.Disk(r, v, p, b, nbt, threshold=(0.0, 50.0, 0.0))
    d.set_precision(prec)
    d.set_gas_grid(*grid)
    assert d.check_ejection_hit_centrum() == len(gone)
    d.handle_ejection_hit_centrum()
    d.clear_event_counter()
    d.rebuild_vectors()
    keep = np.ones(n, bool)
    keep[gone] = False
    r, v, p, b = r[keep], v[keep], p[keep], b[keep]
    want = R.Disk(r, v, p, b, np.bincount(b["body_type"], minlength=7).astype(np.uint32))
    want.set_precision(prec)
    plain = want.calc_dydx(1, 0, 0.0, r, v)
    want.set_gas_grid(*grid)
    got = d.calc_dydx(1, 0, 0.0, r, v)
    assert bits_equal(got, want.calc_dydx(1, 0, 0.0, r, v))
    assert not bits_equal(got, plain)
    # and the grid can still be replaced and removed
    d.set_gas_grid(*fargo_grid(10, 32, 6))
    d.set_gas_grid(None, None, None, None)
    assert bits_equal(d.calc_dydx(1, 0, 0.0, r, v), plain)
