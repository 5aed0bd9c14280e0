"""The direct stages on inputs at the edge of what they accept."""
import numpy as np
import pytest

from vortex_amd import geometry as geo
from vortex_amd.solver import Case, make_params, VX_PREC_F64, VX_PREC_MIXED
from vortex_amd.state import uniform_wake

pytestmark = pytest.mark.gpu
EPS, NU = 0.004, 1e-3


def case(prec, **kw):
    pan = geo.circle(64, 0.5)
    return Case(make_params(pan, precision=prec, ve_size=EPS, nu=NU, **kw), pan)


@pytest.mark.parametrize("prec", [VX_PREC_F64, VX_PREC_MIXED])
@pytest.mark.parametrize("n_src", [0, -1, -1000, -100000])
def test_diffusion_without_sources_adds_nothing(prec, n_src):
    n = 200
    c = case(prec)
    c.set_state(*uniform_wake(n, seed=1))
    u, v, d = np.full(n, 0.25), np.full(n, -0.5), np.full(n, 0.1)
    c.set_velocity(u, v, d)
    c.diffusion(n, n_src)
    got = c.velocity(n)
    c.close()
    for a, b in zip(got, (u, v, d)):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("prec", [VX_PREC_F64, VX_PREC_MIXED])
@pytest.mark.parametrize("n", [500, 20000])
def test_diffusion_threshold_without_bound(prec, n):
    """ve_size has no upper limit; no distance is above an infinite threshold."""
    pan = geo.circle(64, 0.5)
    c = Case(make_params(pan, precision=prec, ve_size=np.inf, nu=NU), pan)
    c.set_state(*uniform_wake(n, seed=2))
    u, v, d = np.full(n, 0.25), np.full(n, -0.5), np.full(n, 0.1)
    c.set_velocity(u, v, d)
    c.diffusion(n, n)
    got = c.velocity(n)
    c.close()
    for a, b in zip(got, (u, v, d)):
        assert np.array_equal(a, b)


def velocity_of(x, y, g, prec=VX_PREC_F64, tree=False):
    n = x.size
    c = case(prec)
    c.set_state(x, y, g)
    if tree:
        c.tree_biot_savart((n + 31) // 32 * 32)
    else:
        c.biot_savart(n, n)
    out = c.velocity(n)
    q = c.velocity_probe(np.linspace(0.6, 4.0, 300), np.linspace(-1.0, 1.0, 300), (0.0, 0.0))
    c.close()
    return out, q


def odd_wake(n, px, py, at=None):
    """A wake and the same with vortices at (px, py); in the first those slots
    are dead and far."""
    x, y, g = uniform_wake(n, seed=n)
    at = np.array([5, n // 2, n - 3][:len(px)])
    x[at], y[at] = 1e10, 1e10
    g0 = g.copy()
    g0[at] = 0.0
    x1, y1 = x.copy(), y.copy()
    x1[at], y1[at] = px, py
    rest = np.ones(n, bool)
    rest[at] = False
    return (x, y, g0), (x1, y1, g), at, rest


@pytest.mark.parametrize("n", [100, 5000, 20000])
@pytest.mark.parametrize("px,py", [((np.nan,), (0.5,)), ((1.0, 1.0), (np.nan, np.nan)), ((np.inf, np.inf), (1.0, 1.0)),
                                   ((-np.inf, np.inf, 2.0), (0.0, 0.0, np.inf))])
def test_sources_without_a_place(n, px, py):
    """Every velocity is NaN then; a NaN or infinite distance is no near one."""
    plain, odd, at, rest = odd_wake(n, px, py)
    (_, _, d0), _ = velocity_of(*plain)
    (u, v, d), q = velocity_of(*odd)
    assert np.all(np.isnan(u)) or np.all(np.isnan(v))
    assert np.array_equal(d[rest], d0[rest])
    # (the padding slots are far, not nowhere)
    np.testing.assert_allclose(d[at], np.sqrt(1e5), rtol=1e-15)
    assert np.all(np.isnan(q[0])) or np.all(np.isnan(q[1]))


@pytest.mark.parametrize("n,tree", [(100, False), (5000, False), (20000, False), (60, True), (300, True)])
@pytest.mark.parametrize("px,py", [((1e200,), (0.0,)), ((1e200, 2e200, -1e180), (0.0, 0.0, 1e190)),
                                   ((1e151, 1.2e151), (3e154, -3e154))])
def test_sources_beyond_the_square_root_of_the_range(n, tree, px, py):
    """Their squared distances are infinite or as good as: they add nothing."""
    plain, odd, at, rest = odd_wake(n, px, py)
    (u0, v0, d0), q0 = velocity_of(*plain, tree=tree)
    (u, v, d), q = velocity_of(*odd, tree=tree)
    tol = 1e-12 if tree else 0.0  # the trees differ
    for a, b in ((u, u0), (v, v0), (d, d0)):
        np.testing.assert_allclose(a[rest], b[rest], rtol=0, atol=tol * np.max(np.abs(b[rest])))
    assert not u[at].any() and not v[at].any()
    np.testing.assert_allclose(d[at], np.sqrt(1e5), rtol=1e-15)
    for a, b in zip(q, q0):
        assert np.array_equal(a, b)
    assert np.all(np.isfinite(q[0]))


@pytest.mark.parametrize("big", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("n,k", [(100, 50), (100, 99), (5000, 7), (5000, 4999), (20000, 123), (20001, 20000)])
def test_circulation_without_bound(n, k, big):
    """Velocities follow its sign (or are NaN); in the diffusion it counts for the
    others alone, whose quotient of sums it makes NaN (or leaves out)."""
    x, y, g = uniform_wake(n, seed=n)
    rest = np.arange(n) != k
    g[k] = big
    (u, v, _), q = velocity_of(x, y, g)
    dx, dy = x - x[k], y - y[k]
    with np.errstate(invalid="ignore"):
        for got, want in ((u, -big * np.sign(dy)), (v, big * np.sign(dx)),
                          (q[0], -big * np.sign(np.linspace(-1.0, 1.0, 300) - y[k])),
                          (q[1], big * np.sign(np.linspace(0.6, 4.0, 300) - x[k]))):
            assert np.array_equal(got, want, equal_nan=True)
    res = []
    for gk in (big, 0.0):
        g[k] = gk
        c = case(VX_PREC_F64)
        c.set_state(x, y, g)
        c.set_velocity(np.full(n, 0.25), np.full(n, -0.5), np.full(n, 0.1))
        c.diffusion(n, n)
        res.append(c.velocity(n)[:2])
        c.close()
    for a, b, z in zip(res[0], res[1], (0.25, -0.5)):
        assert a[k] == b[k] != z
        assert np.all(a[rest] == z) if np.isnan(big) else np.all(np.isnan(a[rest]))
