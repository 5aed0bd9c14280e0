"""The two routes of the mixed-precision birth right-hand side's pairs (up to
32768 sources by terms and ordered adds, above one thread per panel) give the
same bits, as test_gpu_rhs_routes.py checks in FP64."""
import numpy as np
import pytest

from vortex_amd import geometry as geo
from vortex_amd.solver import Case, make_params, VX_PREC_MIXED

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [3, 5, 127, 128, 129, 301])
@pytest.mark.parametrize("n", [1, 64, 127, 129, 255, 257, 512, 513, 3000])
def test_routes_agree(P, n):
    rng = np.random.default_rng(P * 10007 + n)
    r, a = rng.uniform(0.5005, 1.2, n), rng.uniform(0.0, 2 * np.pi, n)
    c = Case(make_params(geo.circle(P, 0.5), precision=VX_PREC_MIXED), geo.circle(P, 0.5))
    c.reserve(33024)
    c.set_state(r * np.cos(a), r * np.sin(a), rng.uniform(-1.0, 1.0, n))
    few = c.right_part(n, (1.0, 0.2))
    many = c.right_part(33024, (1.0, 0.2))
    c.close()
    assert np.all(np.isfinite(few)) and np.array_equal(few, many)
