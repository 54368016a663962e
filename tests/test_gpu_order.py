"""Density order on the device at the edges of the radix sort's tiles (8192
keys, 8 XCD shares): ties by index, zeros, negatives and infinities."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 63, 1025, 8191, 8192, 8193, 70001,
                               1000003])
@pytest.mark.parametrize("f64", [False, True])
def test_density_order(n, f64):
    import torch
    import psod_amd as P
    rng = np.random.default_rng(n)
    rho = np.exp(rng.normal(0, 3, n))
    rho[rng.random(n) < 0.3] = 1.0  # ties
    if not f64:
        rho[rng.random(n) < 0.05] = 0.0
        rho[rng.random(n) < 0.01] = np.inf
        rho[rng.random(n) < 0.01] = -2.0  # counts as 0
    rho = rho.astype(np.float64 if f64 else np.float32)
    ctx = P.default_context()
    f = ctx.density_order_f64 if f64 else ctx.density_order
    isort, nnew = f(torch.from_numpy(rho).cuda())
    key = 1.0 / rho if f64 else -np.maximum(rho, np.float32(0))
    want = np.argsort(key, kind="stable") + 1
    np.testing.assert_array_equal(isort.cpu().numpy(), want)
    assert nnew == min(n, int((rho > 100).sum()) + 1)
