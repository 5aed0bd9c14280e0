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
