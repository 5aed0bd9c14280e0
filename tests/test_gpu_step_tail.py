"""The tail of a step (compaction and collapse passes) as one launch at small
counts gives the same bits as the launches it stands for: stream steps take it
up to 3584 vortices, graph steps of a case with a larger capacity do not.
Crowded and sparse wakes, unequal, equal and zero radii, several passes,
vortices that the move absorbs or deletes, every slot compared (the dead ones
above the count too)."""
import numpy as np
import pytest

from vortex_amd import geometry as geo
from vortex_amd.solver import Case, make_params, VX_PREC_F64

pytestmark = pytest.mark.gpu
VINF = (1.0, 0.0)


def wake(n, crowd, seed):
    rng = np.random.default_rng(seed)
    x, y = rng.uniform(0.6, 0.6 + crowd, n), rng.uniform(-crowd / 2, crowd / 2, n)
    g = rng.uniform(1e-4, 2e-3, n) * rng.choice([-1.0, 1.0], n)
    x[::17] = 9.999  # leaves the box in a step
    g[5::23] = 0.0   # dead before the step
    x[3::41], y[3::41] = rng.uniform(-0.51, -0.505, x[3::41].size), rng.uniform(-0.01, 0.01, y[3::41].size)
    return x, y, g


@pytest.mark.parametrize("n", [0, 1, 2, 63, 900, 1024, 2047, 3400, 3583, 3584])
@pytest.mark.parametrize("crowd,rd,rs,n_col", [(0.05, 1.0, 0.3, 2), (0.4, 0.3, 0.3, 3), (3.0, 2.0, 4.0, 2),
                                               (0.2, 0.0, 1.0, 1), (0.2, 1.0, 1.0, 0)])
def test_one_launch_equals_the_launches(n, crowd, rd, rs, n_col):
    pan = geo.circle(64, 0.5)
    out = []
    for graph in (False, True):
        c = Case(make_params(pan, precision=VX_PREC_F64, dt=0.005, r_col_diff_sign=rd, r_col_same_sign=rs,
                             n_col=n_col, ve_size=0.01, max_ve_g=0.02, birth_offset_rel=0.5), pan)
        c.build_matrix()
        if graph:
            c.reserve(20000)
        c.set_state(*wake(n, crowd, n + 1))
        f = c.run_steps_graph(3, VINF)[0] if graph else c.run_steps(3, VINF)
        slots = (n + 3 * 64 + 31) // 32 * 32
        out.append((c.n, f, *c.state(slots)))
        c.close()
    assert out[0][0] == out[1][0]
    for a, b in zip(out[0][1:], out[1][1:]):
        assert np.array_equal(a, b, equal_nan=True)


def test_captured_step_follows_its_buffers():
    """Calls between two graph runs that grow workspaces or change the form of
    the step leave the second run's results as they were."""
    pan = geo.circle(64, 0.5)
    out = []
    for between in (False, True):
        c = Case(make_params(pan, precision=VX_PREC_F64, dt=0.005, n_col=2, ve_size=0.01, max_ve_g=0.02,
                             birth_offset_rel=0.5), pan)
        c.build_matrix()
        c.set_state(*wake(300, 0.4, 9))
        f = [c.run_steps_graph(3, VINF)[0]]
        if between:
            q = np.random.default_rng(1).uniform(-2.0, 2.0, (2, 60000))
            c.velocity_probe(q[0], q[1], VINF)
        f.append(c.run_steps_graph(3, VINF)[0])
        n = c.n
        c.set_state(*wake(3900, 3.0, 10))  # above the one-launch form
        f.append(c.run_steps_graph(2, VINF)[0])
        f.append(c.run_steps_graph(2, VINF)[0])
        out.append((n, c.n, *f, *c.state(c.n)))
        c.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
