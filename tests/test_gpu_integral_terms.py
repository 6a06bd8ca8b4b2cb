"""A pair term of the energy, m_i m_j / r, is no further from the exact value than
the reference formula's correctly rounded root and division: disks of two
bodies at rest, whose energy is the one term, against 80-bit floats."""
import numpy as np
import pytest

import redamd as R
from systems import small_system

pytestmark = pytest.mark.gpu


def test_two_body_energy_term():
    parts = [small_system(2, 900 + k, spread=5.0) for k in range(2000)]
    for r, v, p, b, nbt in parts:
        for f in "xyz":
            v[f] = 0.0
    d = R.Disk(*[np.concatenate([q[i] for q in parts]) for i in range(4)], np.stack([q[4] for q in parts]),
               batch=True)
    e, ref = [], []
    for k, (r, v, p, b, nbt) in enumerate(parts):
        dx, dy, dz = (r[f][1] - r[f][0] for f in "xyz")
        r2 = dx * dx + dy * dy + dz * dz
        m = p["mass"][0] * p["mass"][1]
        exact = np.longdouble(m) / np.sqrt(np.longdouble(r2))
        ulp = np.spacing(float(exact))
        e.append(float((-d.integral(k)["E"] - exact) / ulp))
        ref.append(float((m / np.sqrt(r2) - exact) / ulp))
    e, ref = np.array(e), np.array(ref)
    # one rounding, and what an 80-bit quotient and a step of 2^-68 leave (2^-10 of a unit)
    assert np.abs(e).max() <= 0.5 + 2.0 ** -10
    assert np.sqrt(np.mean(e * e)) <= np.sqrt(np.mean(ref * ref))
