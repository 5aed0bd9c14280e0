"""Single FP64 pair terms: with every other circulation zero and all vortices on
the x axis, a sum is one term, every operation of which NumPy can repeat, so the
results are compared bit for bit with correctly rounded quotients."""
import numpy as np
import pytest

from vortex_amd import geometry as geo
from vortex_amd.solver import Case, make_params, VX_PREC_F64

pytestmark = pytest.mark.gpu
EPS, NU = 0.004, 1e-3


def line(n, seed):
    """n vortices on the axis; the first alone has circulation."""
    rng = np.random.default_rng(seed)
    x = rng.uniform(1.0, 9.0, n)
    g = np.zeros(n)
    g[0] = rng.uniform(0.001, 0.004)
    pan = geo.circle(64, 0.5)
    c = Case(make_params(pan, precision=VX_PREC_F64, ve_size=EPS, nu=NU), pan)
    c.set_state(x, np.zeros(n), g)
    return c, x, g[0]


def biot_savart_v(x, x0, g):
    dx = x - x0
    return g / np.maximum(dx * dx, EPS * EPS) * dx / (2 * np.pi)


@pytest.mark.parametrize("n", [20000, 40000])
def test_split_biot_savart(n):
    c, x, g = line(n, n)
    c.biot_savart(n, n)
    v = c.velocity(n)[1]
    c.close()
    assert np.array_equal(v, biot_savart_v(x, x[0], g))


def test_probe():
    c, x, g = line(32, 3)
    px = np.random.default_rng(4).uniform(0.0, 10.0, 20000)
    v = c.velocity_probe(px, np.zeros(px.size), (0.0, 0.0))[1]
    c.close()
    assert np.array_equal(v, biot_savart_v(px, x[0], g))


@pytest.mark.parametrize("n", [33, 64])
def test_tree_near_pairs(n):
    """One bucket holds all, so that every pair is a near one."""
    for seed in range(40):
        c, x, g = line(n, 100 * n + seed)
        c.tree_biot_savart((n + 31) // 32 * 32)
        v = c.velocity(n)[1]
        c.close()
        assert np.array_equal(v, biot_savart_v(x, x[0], g))


def diffusion_u(x, x0, g, d):
    """One term whose exponential is 1 (d far above the separations)."""
    dx = x - x0
    r = np.abs(dx)
    on = r > 0.001 * EPS
    w = g / np.where(on, r, 1.0)
    return np.where(on, NU * (w * dx) / (g * d), 0.0)


@pytest.mark.parametrize("n,tree", [(20000, False), (40001, False), (5000, False), (64, True), (4000, True)])
def test_diffusion(n, tree):
    c, x, g = line(n, n)
    c.biot_savart(n, n)
    if tree:
        c.tree_biot_savart((n + 31) // 32 * 32)
    z, d = np.zeros(n), np.full(n, 1e30)
    c.set_velocity(z, z, d)
    if tree:
        c.tree_diffusion()
    else:
        c.diffusion(n, n)
    u, v, _ = c.velocity(n)
    c.close()
    assert np.array_equal(u, diffusion_u(x, x[0], g, d)) and not v.any()


@pytest.mark.parametrize("d", [0.01, 1e30])
@pytest.mark.parametrize("n,tree", [(100, False), (20000, False), (40001, False), (100, True), (6000, True)])
def test_diffusion_threshold(n, tree, d):
    """Separations of one unit of rounding, and of more, on both sides of the
    threshold of 0.001 ve_size: a pair counts above it alone."""
    pan = geo.circle(64, 0.5)
    thr = 0.001 * EPS
    sep = np.array([0.5 * thr, np.nextafter(thr, 0.0), thr, np.nextafter(thr, 1.0), 1.5 * thr, 1.999 * thr, 3.0 * thr])
    rng = np.random.default_rng(n)
    x, g = rng.uniform(1.0, 9.0, n), np.zeros(n)
    x[0], g[0] = 0.0, 0.002
    at = np.r_[1:8, n - 8:n - 1]
    x[at] = np.r_[sep, -sep]
    c = Case(make_params(pan, precision=VX_PREC_F64, ve_size=EPS, nu=NU), pan)
    c.set_state(x, np.zeros(n), g)
    if tree:
        c.tree_biot_savart((n + 31) // 32 * 32)
    z, dd = np.zeros(n), np.full(n, d)
    c.set_velocity(z, z, dd)
    if tree:
        c.tree_diffusion()
    else:
        c.diffusion(n, n)
    u = c.velocity(n)[0]
    c.close()
    on = np.abs(x[at]) > thr
    assert on.sum() == 8
    assert u[0] == 0.0 and not u[at][~on].any()
    # the exponential stands in both sums and leaves the quotient
    np.testing.assert_allclose(u[at][on], (NU * np.sign(x[at]) / d)[on], rtol=1e-14)
