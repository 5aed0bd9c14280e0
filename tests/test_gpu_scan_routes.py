"""Hit panels, wall term and birth right-hand side of small counts without
lists or with fewer launches, against the routes of larger bounds, bit for
bit: the same captured steps with the case's own capacity (within 32768 and, for
the right-hand side, 8192) and with a larger one."""
import numpy as np
import pytest

from vortex_amd import geometry as geo
from vortex_amd.solver import Case, make_params, VX_PREC_F64, VX_PREC_MIXED

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [VX_PREC_F64, VX_PREC_MIXED])
@pytest.mark.parametrize("n,P,points", [(0, 64, 20), (1, 3, 7), (255, 65, 20), (4095, 200, 64), (4097, 257, 20),
                                        (7000, 129, 30)])
def test_steps(n, P, points, prec):
    pan = geo.circle(P, 0.5)
    out = []
    for cap in (0, 40000):
        c = Case(make_params(pan, precision=prec, dt=0.02, n_col=1, ve_size=0.004, birth_offset_rel=0.5,
                             n_of_points=points), pan)
        c.build_matrix()
        c.reserve(cap)
        rng = np.random.default_rng(n + P)
        # a ring close to the profile: many candidates, some absorbed, most in the wall's box
        r, a = 0.502 + 0.2 * rng.random(n) ** 2, rng.uniform(0.0, 2 * np.pi, n)
        c.set_state(r * np.cos(a), r * np.sin(a), rng.uniform(-0.02, 0.02, n))
        f, counts = c.run_steps_graph(2, (1.0, 0.1))
        out.append((counts, f, *c.state(int(counts[-1]))))
        c.close()
    for p, q in zip(*out):
        assert np.array_equal(p, q, equal_nan=True)
    if n >= 4095:
        assert out[0][0][0] < n + P  # some were absorbed


@pytest.mark.parametrize("prec", [VX_PREC_F64, VX_PREC_MIXED])
@pytest.mark.parametrize("n", [300, 8192])
def test_right_part_routes(n, prec):
    pan = geo.circle(301, 0.5)
    c = Case(make_params(pan, precision=prec), pan)
    c.reserve(33024)
    rng = np.random.default_rng(n)
    r, a = rng.uniform(0.501, 3.0, n), rng.uniform(0.0, 2 * np.pi, n)
    c.set_state(r * np.cos(a), r * np.sin(a), rng.uniform(-1.0, 1.0, n))
    R = [c.right_part(k, (1.0, 0.2)) for k in (n, 8224, 20000, 32768, 33024)]
    c.close()
    assert np.all(np.isfinite(R[0]))
    for q in R[1:]:
        assert np.array_equal(R[0], q)
