"""More quadrature points a panel than 2^24: every one is taken.  In FP64 the
result hardly depends on so many, but FP32 sums end where a term falls below
their last digit, so their value tells the count: 2^26 points and 2^24 differ by
half.  The reference repeats the sums one by one in NumPy's FP32; it rounds the
products, which the kernel's fused operations do not, hence 5 %."""
import numpy as np
import pytest

from vortex_amd import geometry as geo
from vortex_amd.solver import Case, make_params, VX_PREC_MIXED

pytestmark = pytest.mark.gpu
X, Y, D = 0.9, 0.13, 0.2


def fp32_wall(pan, points):
    """II3 / II0 at (X, Y) over the panels in range, as src/kernel.cu:1031-1088."""
    f, i0, i3 = np.float32, 2 * np.pi * D * D, np.zeros(2)
    k = np.arange(points, dtype=f)
    for p in pan:
        if not 0.1 * p["length"] < np.hypot(*(p["birth"] - (X, Y))) < 5 * p["length"]:
            continue
        ra, rb, n = ((a).astype(f) for a in (p["left"] - (X, Y), p["right"] - (X, Y), -p["norm"]))
        step, width = (rb - ra) / f(points), f(p["length"]) / f(points)
        e = [-(ra[c] + (k + f(0.5)) * step[c]) / f(D) for c in range(2)]
        e2 = e[0] * e[0] + e[1] * e[1]
        r = np.sqrt(e2)
        ex = np.exp(-r)
        s = [np.add.accumulate(width * t, dtype=f)[-1]
             for t in ((e[0] * n[0] + e[1] * n[1]) / e2 * (r + f(1)) * ex, n[0] * ex, n[1] * ex)]
        i0 -= D * float(s[0])
        i3 += s[1:]
    return i3 / i0


@pytest.mark.parametrize("points", [1 << 24, 1 << 26])
def test_fp32_sums_of_many_points(points):
    pan = geo.circle(4, 0.5)
    c = Case(make_params(pan, precision=VX_PREC_MIXED, nu=1.0, n_of_points=points), pan)
    c.set_state(np.array([X]), np.array([Y]), np.array([0.01]))
    c.set_velocity(np.zeros(1), np.zeros(1), np.array([D]))
    c.diffusion_wall(1)
    u, v, _ = c.velocity(1)
    c.close()
    want = -fp32_wall(pan, points)
    print(f"[wall] {points} points: {u[0]} {v[0]}, expected {want}", flush=True)
    np.testing.assert_allclose([u[0], v[0]], want, rtol=0.05)
