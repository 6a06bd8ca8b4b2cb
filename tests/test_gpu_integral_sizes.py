"""The integrals' block edges (256 sinks, 128 sources, single bodies) against
plain FP64 sums, with inactive bodies and masses outside the short root and
division sequences."""
import math

import numpy as np
import pytest

import redamd as R
from systems import small_system, as3

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("odd", [False, True])
@pytest.mark.parametrize("n", [1, 2, 127, 128, 129, 256, 257, 385, 1030])
def test_integral_block_edges(n, odd):
    inactive = tuple(range(3, n, 50))
    r, v, p, b, nbt = small_system(n, 500 + n, inactive=inactive)
    if odd and n > 2:
        p["mass"][2] = 1e-95
    q = R.Disk(r, v, p, b, nbt).integral()
    on = b["id"] > 0
    x, u, m = as3(r)[on], as3(v)[on], p["mass"][on]
    d = np.sqrt(((x[:, None] - x[None]) ** 2).sum(-1))
    pair = (m[:, None] * m[None] / np.where(d > 0, d, np.inf))[np.triu_indices(len(m), 1)]
    kin = math.fsum(m * (u * u).sum(1)) / 2.0
    pot = math.fsum(pair)
    # a pair term is within 3 ulp of the numpy one (distance, root, product and
    # division each rounded), the sums are exact to an ulp
    assert abs(q["E"] - (kin - pot)) <= 4 * 2.0 ** -52 * (kin + pot)
    c = np.cross(x, u) * m[:, None]
    for k, f in enumerate("xyz"):
        s = np.abs(c[:, k]).sum() + 1e-300
        assert abs(q["C"][f] - math.fsum(c[:, k])) <= 4 * 2.0 ** -52 * s
        assert abs(q["R"][f] - math.fsum(m * x[:, k]) / m.sum()) <= 4 * 2.0 ** -52 * np.abs(m * x[:, k]).sum() / m.sum()
