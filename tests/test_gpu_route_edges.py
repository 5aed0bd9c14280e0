"""Routes at the counts where they change: the selection as one work-group (up to
32768 items), through the callers that take it, and the last sums of the
diffusion's domain-scale targets, eight a work-group."""
import numpy as np
import pytest

import test_gpu_tree_far
from vortex_amd import geometry as geo
from vortex_amd.solver import Case, make_params, VX_PREC_F64, VX_PREC_MIXED
from vortex_amd.state import uniform_wake

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [992, 1024, 1056, 32736, 32768, 32800])
def test_wall_list_beside_the_diffusion(n):
    """The velocity stage lists the wall's targets for the second stream; the wall
    pass by itself scans them without a list up to 32768.  (The larger wakes hold
    coincident vortices, whose d is 0 and whose wall term is NaN in both.)"""
    pan = geo.circle(200, 0.5)
    x, y, g = uniform_wake(n, seed=n)
    x[::50] = 0.51 + 0.001 * (np.arange(x[::50].size) % 7)
    y[::50] = 0.001 * (np.arange(y[::50].size) % 11)
    out = []
    for stages in (False, True):
        c = Case(make_params(pan, precision=VX_PREC_F64, nu=1e-3, ve_size=0.004), pan)
        c.set_state(x, y, g)
        if stages:
            c.biot_savart(n, n, (1.0, 0.0))
            c.diffusion(n, n)
            before = c.velocity(n)[0]
            c.diffusion_wall(n)
        else:
            c.speed((1.0, 0.0))
        out.append(c.velocity(n))
        c.close()
    assert np.count_nonzero(out[1][0] != before) > n // 100
    for a, b in zip(*out):
        assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("near", [0, 1])
@pytest.mark.parametrize("n", [1023, 1024, 1025, 32767, 32768, 32769])
def test_near_source_list(n, near):
    """The birth's right-hand side over n sources and over the same with an empty
    far tail, whose list comes from several work-groups."""
    rng = np.random.default_rng(n + near)
    r, a = rng.uniform(0.501, 0.99 if near else 6.0, n), rng.uniform(0.0, 2 * np.pi, n)
    pan = geo.circle(200, 0.5)
    c = Case(make_params(pan, precision=VX_PREC_F64), pan)
    c.reserve(131104)
    c.set_state(r * np.cos(a), r * np.sin(a), rng.uniform(-1.0, 1.0, n))
    few, many = c.right_part(n, (1.0, 0.2)), c.right_part(131104, (1.0, 0.2))
    c.close()
    assert np.all(np.isfinite(few)) and np.array_equal(few, many)


@pytest.mark.parametrize("prec,tol", [(VX_PREC_F64, 1e-9), (VX_PREC_MIXED, 1e-3)])
@pytest.mark.parametrize("k", [7, 8, 9])
def test_isolated_targets_at_the_tiles(k, prec, tol):
    test_gpu_tree_far.test_isolated_targets(6000, k, prec, tol)
