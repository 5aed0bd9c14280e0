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
