"""The wall term's quadrature with its points dealt over the wave: panel counts
around the wave and the group of four rounds, point counts around and above
64, panels that all lie in range, targets that a first panel decides alone.
Tolerances as in test_gpu_parity.py: 1e-12 of the largest value in FP64, 5e-4
in mixed precision."""
import numpy as np
import pytest

from vortex_amd import geometry as geo
from vortex_amd.solver import Case, make_params, VX_PREC_F64, VX_PREC_MIXED

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,tol", [(VX_PREC_F64, 1e-12), (VX_PREC_MIXED, 5e-4)])
@pytest.mark.parametrize("points", [1, 7, 20, 63, 64, 65, 130])
@pytest.mark.parametrize("P", [3, 5, 63, 64, 65, 255, 256, 257, 520])
def test_wall(ref, P, points, prec, tol):
    pan = geo.circle(P, 0.5)
    c = Case(make_params(pan, precision=prec, nu=1e-3, n_of_points=points), pan)
    rng = np.random.default_rng(P * 1000 + points)
    n, dl = 200, float(pan["length"].mean())
    th, r = rng.uniform(0, 2 * np.pi, n), 0.5 + dl * rng.uniform(0.0, 5.5, n)
    x, y = r * np.cos(th), r * np.sin(th)
    k = rng.integers(0, P, 20)  # within 0.1 l of a birth point
    x[:20], y[:20] = pan["birth"][k, 0] + 0.03 * dl, pan["birth"][k, 1] - 0.02 * dl
    d = dl * rng.uniform(0.3, 3.0, n)
    c.set_state(x, y, rng.uniform(-0.01, 0.01, n))
    c.set_velocity(np.zeros(n), np.zeros(n), d)
    c.diffusion_wall(n)
    u, v, _ = c.velocity(n)
    c.close()
    ur, vr = ref.diffusion_wall(x, y, d, pan, 1e-3, points)
    scale = max(np.abs(ur).max(), np.abs(vr).max())
    assert scale > 0
    assert np.max(np.abs(u - ur)) < tol * scale and np.max(np.abs(v - vr)) < tol * scale
