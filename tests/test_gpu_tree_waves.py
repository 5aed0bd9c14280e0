"""The tree's velocity stages with several waves a target group (diffusion) or
bucket (Biot-Savart up to 14336 buckets in FP64, 8192 in mixed precision):
edges of the groups, pairs around the diffusion's threshold, and counts on both
sides of the limits.
Tolerances as stated in test_gpu_tree.py: diffusion FP64 1e-9, mixed 1e-3 (one
sign of circulation, so the weight sums do not cancel); Biot-Savart FP64 with
32 terms 1e-8, mixed with 16 terms 3e-4 (nearest-3 distance 1e-4)."""
import numpy as np
import pytest

from vortex_amd import geometry as geo
from vortex_amd.solver import Case, make_params, VX_PREC_F64, VX_PREC_MIXED

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,tol", [(VX_PREC_F64, 1e-9), (VX_PREC_MIXED, 1e-3)])
@pytest.mark.parametrize("n", [4, 33, 63, 64, 65, 129, 257, 1000, 6000])
def test_diffusion_small_sizes(ref, n, prec, tol):
    rng = np.random.default_rng(n)
    x, y = rng.uniform(1.0, 2.0, n), rng.uniform(-0.5, 0.5, n)
    g = rng.uniform(0.001, 0.004, n)
    eps, nu = 0.004, 1e-3
    if n > 60:  # coincident, below the threshold of 0.001 eps, above it
        x[1:4], y[1:4] = x[0], y[0] + np.array([0.0, 0.0005, 0.003]) * eps
    pan = geo.circle(64, 0.5)
    c = Case(make_params(pan, precision=prec, ve_size=eps, nu=nu), pan)
    s = (n + 31) // 32 * 32
    c.set_state(x, y, g)
    c.tree_biot_savart(s, (0.0, 0.0))
    X, Y, G = c.state(s)
    u0, v0, d = c.velocity(s)
    c.tree_diffusion()
    u, v, _ = c.velocity(s)
    c.close()
    ur, vr = ref.diffusion(X, Y, G, d, nu, eps, u0, v0)
    if n > 60:  # their own d is of rounding size, their weights far below the sums' cut
        assert np.all(np.isfinite(u)) and np.all(np.isfinite(v))
    far = np.arange(n) >= 4 if n > 60 else np.ones(n, bool)
    for a, b, z in ((u, ur, u0), (v, vr, v0)):
        e, r = (a - z)[:n][far], (b - z)[:n][far]
        assert np.max(np.abs(e - r)) <= tol * np.max(np.abs(r))


@pytest.mark.parametrize("n", [560000, 700000])
def test_biot_savart_around_the_split_limit(n):
    """Against the direct sums at every thousandth vortex (the probe's own pair
    adds nothing)."""
    rng = np.random.default_rng(n)
    x, y = rng.uniform(0.7, 9.5, n), rng.uniform(-4.0, 4.0, n)
    g = rng.uniform(-0.004, 0.004, n)
    pan = geo.circle(64, 0.5)
    c = Case(make_params(pan, precision=VX_PREC_F64, ve_size=0.004, order=32), pan)
    c.set_state(x, y, g)
    c.tree_biot_savart((n + 31) // 32 * 32, (0.0, 0.0))
    u, v, _ = c.velocity(n)
    assert (c.tree_stats()["leaves"] > 14336) == (n == 700000)
    k = np.arange(0, n, 1000)
    up, vp = c.velocity_probe(x[k], y[k], (0.0, 0.0))
    c.close()
    for a, b in ((u[k], up), (v[k], vp)):
        assert np.max(np.abs(a - b)) <= 1e-8 * np.max(np.abs(b))


@pytest.mark.parametrize("n", [250000, 700000])
def test_biot_savart_mixed_around_the_split_limit(n):
    """The same for the mixed tree; the nearest-3 distances against the FP64
    tree's, whose searches are exact."""
    rng = np.random.default_rng(n)
    x, y = rng.uniform(0.7, 9.5, n), rng.uniform(-4.0, 4.0, n)
    g = rng.uniform(-0.004, 0.004, n)
    pan = geo.circle(64, 0.5)
    res = {}
    for prec in (VX_PREC_MIXED, VX_PREC_F64):
        c = Case(make_params(pan, precision=prec, ve_size=0.004, order=16), pan)
        c.set_state(x, y, g)
        c.tree_biot_savart((n + 31) // 32 * 32, (0.0, 0.0))
        res[prec] = c.velocity(n)
        assert (c.tree_stats()["leaves"] > 8192) == (n == 700000)
        if prec == VX_PREC_F64:
            k = np.arange(0, n, 1000)
            up, vp = c.velocity_probe(x[k], y[k], (0.0, 0.0))
        c.close()
    u, v, d = res[VX_PREC_MIXED]
    for a, b in ((u[k], up), (v[k], vp)):
        assert np.max(np.abs(a - b)) <= 3e-4 * np.max(np.abs(b))
    np.testing.assert_allclose(d, res[VX_PREC_F64][2], rtol=1e-4, atol=0)
