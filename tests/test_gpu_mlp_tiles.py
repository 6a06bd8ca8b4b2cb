"""The gradient kernel's block edges (64 samples in 16-row tiles) and the
partials' reduction (64 at a time) against the float64 reference."""
import numpy as np
import pytest

import mlp_ref as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("quantile", [0.0, 0.05])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 4095, 4097, 8200])
def test_gradient_block_edges(n, quantile):
    import redamd as R
    rng = np.random.default_rng(n)
    w = rng.normal(0, 0.3, M.NPARAM).astype(np.float32)
    mean = rng.normal(0, 1, M.IN).astype(np.float32)
    std = rng.uniform(0.5, 2.0, M.IN).astype(np.float32)
    m = R.Mlp(1)
    m.set_params(w)
    m.set_norm(mean, std, 0.3, 1.7)
    m.set_target(9, quantile)
    x = rng.normal(0, 2, (n, M.IN)).astype(np.float32)
    t = (x[:, 9] + rng.normal(0, 1, n)).astype(np.float32)
    loss, g = m.loss_grad(x, t)
    loss_ref, g_ref = M.loss_grad(w, x, t, mean.astype(np.float64), std.astype(np.float64), 0.3, 1.7, 9, quantile)
    # FP32 throughout, chains of at most 64 terms and then the blocks: relative to
    # the largest entry of each parameter block, as the other gradient tests
    assert abs(loss - loss_ref) <= 1e-5 * abs(loss_ref)
    k = 0
    for name, size in M.SIZES:
        ref = g_ref[k:k + size]
        assert np.max(np.abs(g[k:k + size] - ref)) <= 1e-4 * np.max(np.abs(ref)), name
        k += size
