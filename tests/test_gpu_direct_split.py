"""Work split of the direct kernels (vx_biot_savart, vx_diffusion): counts at
the edges of the ordered FP64 kernels' tiles (16 or 32 targets, 120 or 60
sources), of the FP32 tiles (256 sources) and of the bound between ordered and
split FP64 sums (16384 sources), against the FP64 oracle.

Tolerances: a sum of n terms added one by one, or in runs, is off by at most
(n + c) u times the sum of the terms' magnitudes, with u the unit roundoff
and c u the error of a term itself; FP32 terms are added in FP32 over 256
sources and in FP64 beyond, so n is 256 there.  The oracle gets the FP32
coordinates, which leaves the arithmetic's error alone."""
import numpy as np
import pytest

from vortex_amd import geometry as geo
from vortex_amd.solver import Case, make_params, VX_PREC_F64, VX_PREC_MIXED
from vortex_amd.state import uniform_wake

pytestmark = pytest.mark.gpu
EPS, NU = 0.004, 1e-3


def magnitudes(x, y, g, rows):
    """Per target: sums of |g|/r-like terms, squared distances."""
    dx = x[rows, None] - x[None, :]
    dy = y[rows, None] - y[None, :]
    r2 = dx * dx + dy * dy
    return dx, dy, r2, np.abs(g) / np.maximum(r2, EPS * EPS)


@pytest.mark.parametrize("prec", [VX_PREC_F64, VX_PREC_MIXED])
@pytest.mark.parametrize("n", [1, 31, 64, 119, 120, 121, 255, 257, 1000, 4095, 4097, 16384, 16385, 16500])
def test_direct_sums_at_the_edges(ref, prec, n):
    x, y, g = uniform_wake(n, seed=n)
    f32 = prec == VX_PREC_MIXED
    if f32:
        x, y, g = (a.astype(np.float32).astype(np.float64) for a in (x, y, g))
    pan = geo.circle(64, 0.5)
    c = Case(make_params(pan, precision=prec, ve_size=EPS, nu=NU), pan)
    c.set_state(x, y, g)
    m = max(1, n - 3)  # fewer targets than sources
    c.biot_savart(m, n, (1.0, 0.0))
    u, v, d = c.velocity(m)
    ur, vr, dr = ref.biot_savart(x, y, g, EPS * EPS, (1.0, 0.0), n_tgt=m)
    rows = np.unique(np.r_[0:min(m, 96), max(0, m - 96):m])
    dx, dy, r2, w = magnitudes(x, y, g, rows)
    unit = 2.0 ** -24 if f32 else 2.0 ** -53
    terms = (min(n, 256) if f32 else n) + 24
    for got, want, q in ((u, ur, dy), (v, vr, dx)):
        bound = terms * unit * np.sum(w * np.abs(q), axis=1) / (2 * np.pi) + 4 * 2.0 ** -53 * np.abs(want[rows])
        assert np.all(np.abs(got[rows] - want[rows]) <= bound)
    assert np.all(np.abs(d - dr[:m]) <= 8 * unit * dr[:m])
    # diffusion over the same d
    c.set_velocity(np.zeros(m), np.zeros(m), dr[:m])
    c.diffusion(m, n)
    u, v, _ = c.velocity(m)
    ur, vr = ref.diffusion(x, y, g, dr, NU, EPS, np.zeros(n), np.zeros(n), n_tgt=m)
    r = np.sqrt(r2)
    on = r > 1e-3 * EPS
    e = np.where(on, np.exp(-r / dr[rows, None]), 0.0)
    # a term's exponent is off by a few units of itself
    rel = (terms + 4 * r / dr[rows, None]) * unit
    i1 = np.sum(g * e, axis=1)
    d1 = np.sum(rel * np.abs(g) * e, axis=1)
    sure = np.abs(np.abs(i1) - 1e-5) > 4 * d1
    for got, want, q in ((u, ur, dx), (v, vr, dy)):
        t = np.where(on, g * e * q / np.where(on, r, 1.0), 0.0)
        i2, d2 = np.abs(np.sum(t, axis=1)), np.sum(rel * np.abs(t), axis=1)
        with np.errstate(divide="ignore", invalid="ignore"):
            bound = np.where(np.abs(i1) > 1e-5,
                             NU / dr[rows] * (d2 + i2 * d1 / np.abs(i1)) / (np.abs(i1) - d1).clip(1e-6) * 2, 0.0)
        bound = bound + 4 * 2.0 ** -53 * np.abs(want[rows])
        assert np.all((np.abs(got[rows] - want[rows]) <= bound)[sure])
    c.close()


@pytest.mark.parametrize("prec", [VX_PREC_F64, VX_PREC_MIXED])
@pytest.mark.parametrize("n", [15000, 16300])
def test_graph_steps_across_the_ordered_bound(prec, n):
    """Graph replays whose capacity lies above 16384 sources while the count
    stays below it, or passes it, equal stream steps bit for bit."""
    pan = geo.circle(128, 0.5)
    out = []
    for graph in (False, True):
        c = Case(make_params(pan, precision=prec, dt=0.005, nu=NU, r_col_diff_sign=0.3, r_col_same_sign=0.3,
                             birth_offset_rel=0.5), pan)
        c.build_matrix()
        c.reserve(24000)
        c.set_state(*uniform_wake(n, seed=4, max_ve_g=1e-4))
        f = c.run_steps_graph(4, (1.0, 0.0))[0] if graph else c.run_steps(4, (1.0, 0.0))
        out.append((c.n, f, *c.state()))
        c.close()
    assert out[0][0] == out[1][0]
    for a, b in zip(out[0][1:], out[1][1:]):
        assert np.array_equal(a, b)
