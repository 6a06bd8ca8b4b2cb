"""Mixed precision: the sums over a chunk of one-sided sources stay FP64 where the
chunk is cut into 256-source tiles.  Two heavy sources pull a sink in opposite
directions, one tile apart, beside a light one: rounding a tile's sum to FP32
would leave 2^-24 of the heavy pull, 1/16 of the light one."""
import numpy as np
import pytest

import redamd as R
from redamd_types import VAR4, PARAM, BODY_MD

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sinks", [1, 2, 4])
@pytest.mark.parametrize("sink,source", [(6, 3), (5, 3), (3, 5)])
def test_cut_chunk_sums(sink, source, sinks):
    n_src = 1000
    types = [0] + ([sink] + [source] * n_src if sink < source else [source] * n_src + [sink])
    n = len(types)
    i, j0 = (1, 2) if sink < source else (n - 1, 1)   # the sink, the first source
    rng = np.random.default_rng(3)
    r, v, p, b = np.zeros(n, VAR4), np.zeros(n, VAR4), np.zeros(n, PARAM), np.zeros(n, BODY_MD)
    for f in "xyz":
        r[f] = rng.uniform(0.1, 2.0, n)
    b["body_type"], b["id"] = types, np.arange(1, n + 1)
    p["radius"], p["density"] = 1e-5, 1e6
    # all other masses are zero, the star's too
    heavy, light, mirror = j0, j0 + 64, j0 + 256     # two quarters of a tile, and the next tile
    for k, m, at in ((heavy, 2.0 ** -10, (0.6, 0.8, 0.1)), (light, 2.0 ** -30, (0.3, -0.9, 0.2)),
                     (mirror, 2.0 ** -10, (-0.6, -0.8, -0.1))):
        p["mass"][k] = m
        r["x"][k], r["y"][k], r["z"][k] = at
    for f in "xyz":
        r[f][i] = 0.0
    d = R.Disk(r, v, p, b, np.bincount(types, minlength=7).astype(np.uint32))
    d.set_precision(R.RD_PREC_MIXED)
    d.set_tuning(sinks_per_lane=sinks)
    a = d.calc_dydx(1, 0, 0.0, r, v)[i]
    x = np.array([0.3, -0.9, 0.2])
    want = 2.0 ** -30 * x / np.sqrt(x @ x) ** 3
    got = np.array([a["x"], a["y"], a["z"]])
    # the light term's FP32 operations (offset, r^2, 1.5 ulp rsqrt cubed, product): below 2^-20
    assert np.all(np.abs(got - want) <= 2.0 ** -20 * np.abs(want))
