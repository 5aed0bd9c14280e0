"""The diffusion's domain-scale targets: a dense cloud with k isolated vortices
around it, all of which are listed (and, where the line is low against the
cloud's spacing, a few of its rim).  k at the edges of the kernels' tiles (16
targets a work-group in the last, 64 a wave in the list's), and clouds of few
chunks, of more than 64 (a second mask word) and of more than 256 (a second
pass over the slots).  Against the direct sums at the isolated targets;
tolerances as stated in test_gpu_tree.py: FP64 1e-9, mixed 1e-3 (one sign of
circulation, so the weight sums do not cancel)."""
import numpy as np
import pytest

from vortex_amd import geometry as geo
from vortex_amd.solver import Case, make_params, VX_PREC_F64, VX_PREC_MIXED

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,tol", [(VX_PREC_F64, 1e-9), (VX_PREC_MIXED, 1e-3)])
@pytest.mark.parametrize("n,k", [(6000, 1), (6000, 15), (6000, 16), (6000, 17), (6000, 64), (6000, 65),
                                 (300000, 33), (1200000, 17)])
def test_isolated_targets(n, k, prec, tol):
    rng = np.random.default_rng(n + k)
    x, y = rng.uniform(1.0, 3.0, n), rng.uniform(-1.0, 1.0, n)
    a = 2.0 * np.pi * (np.arange(k) + rng.uniform(-0.2, 0.2, k)) / k
    rad = rng.uniform(11.0, 13.0, k)
    x, y = np.append(x, 2.0 + rad * np.cos(a)), np.append(y, rad * np.sin(a))
    g = rng.uniform(0.001, 0.004, n + k)
    eps, nu = 0.004, 1e-3
    pan = geo.circle(64, 0.5)
    c = Case(make_params(pan, precision=prec, ve_size=eps, nu=nu), pan)
    c.set_state(x, y, g)
    c.tree_biot_savart((n + k + 31) // 32 * 32, (0.0, 0.0))
    u0, v0, d = c.velocity(n + k)
    c.tree_diffusion()
    u, v, _ = c.velocity(n + k)
    st = c.tree_stats()
    c.close()
    assert k <= st["heavy"] < 4096
    chunks = (st["leaves"] + 63) // 64
    assert chunks <= 64 if n == 6000 else chunks > (256 if n == 1200000 else 64)
    ur, vr = np.zeros(k), np.zeros(k)
    for q, i in enumerate(range(n, n + k)):
        dx, dy = x[i] - x, y[i] - y
        r = np.hypot(dx, dy)
        far = r > 0.001 * eps
        w = g[far] * np.exp(-r[far] / d[i])
        s1 = np.sum(w)
        if abs(s1) > 1e-5:
            ur[q] = nu * np.sum(w * dx[far] / r[far]) / (s1 * d[i])
            vr[q] = nu * np.sum(w * dy[far] / r[far]) / (s1 * d[i])
    for b, z, e in ((u, u0, ur), (v, v0, vr)):
        assert np.max(np.abs((b - z)[n:] - e)) <= tol * np.max(np.abs(e))
