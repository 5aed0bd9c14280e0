"""The merge search over crowded cells (long lists in all four cells of a
vortex, lists of very different length, none at all) and the compaction around
the edges of tiles and of its one-launch form (32768 slots), against the oracle,
and steps in both forms of a pass against each other, bit for bit."""
import numpy as np
import pytest

from vortex_amd import geometry as geo
from vortex_amd.solver import Case, make_params, VX_PREC_F64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 300, 4095, 4097, 9000])
@pytest.mark.parametrize("size", [1e-9, 0.004, 0.02, 1.0])
@pytest.mark.parametrize("kind", [1, 2])
def test_search(ref, n, size, kind):
    rng = np.random.default_rng(n)
    x, y = rng.normal(0.0, size, n) + 2.0, rng.normal(0.0, size, n)
    g = rng.uniform(1e-4, 2e-3, n) * rng.choice([-1.0, 1.0], n)
    g[::7] = 0.0
    pan = geo.circle(8, 0.5)
    prm = make_params(pan, precision=VX_PREC_F64, ve_size=0.004, r_col_diff_sign=1.0, r_col_same_sign=0.6, max_ve_g=3e-3)
    c = Case(prm, pan)
    c.set_state(x, y, g)
    col = c.setka(kind)
    r = prm.r_col_diff_sign if kind == 1 else prm.r_col_same_sign
    r2 = r * r * (prm.ve_size * prm.ve_size)
    assert np.array_equal(col, ref.setka(x, y, g, kind, r2, prm.max_ve_g))
    c.close()


@pytest.mark.parametrize("n", [4095, 8192, 8193, 12288, 20481, 32767, 32768, 32769])
@pytest.mark.parametrize("dead", [0.02, 0.4, 0.98])
def test_compaction_around_tile_edges(ref, n, dead):
    rng = np.random.default_rng(n)
    x, y, g = rng.normal(size=n), rng.normal(size=n), rng.uniform(0.1, 1.0, n)
    g[rng.random(n) < dead] = 0.0
    g[-3:] = 0.0, 1.0, 0.0
    pan = geo.circle(8, 0.5)
    c = Case(make_params(pan, precision=VX_PREC_F64), pan)
    c.set_state(x, y, g)
    c.compact()
    xr, yr, gr, nr = ref.compact(x, y, g)
    assert c.n == nr
    for a, b in zip(c.state(n), (xr, yr, gr)):
        assert np.array_equal(a, b)
    c.close()


@pytest.mark.parametrize("n", [3600, 8000, 32300])
def test_passes_in_one_launch(n):
    """A pass whose compaction follows in the same launch (the count's bound
    within 32768) against the one that launches it apart."""
    pan = geo.circle(64, 0.5)
    out = []
    for cap in (0, 60000):
        c = Case(make_params(pan, precision=VX_PREC_F64, dt=0.005, r_col_diff_sign=1.0, r_col_same_sign=0.5, n_col=2,
                             ve_size=0.01, max_ve_g=0.02, birth_offset_rel=0.5), pan)
        c.build_matrix()
        c.reserve(cap)
        rng = np.random.default_rng(n)
        x, y = rng.uniform(0.6, 1.6, n), rng.uniform(-0.5, 0.5, n)
        c.set_state(x, y, rng.uniform(1e-4, 2e-3, n) * rng.choice([-1.0, 1.0], n))
        f = c.run_steps_graph(2, (1.0, 0.0))[0]
        out.append((c.n, f, *c.state(n)))
        c.close()
    assert out[0][0] == out[1][0] < n
    for a, b in zip(out[0][1:], out[1][1:]):
        assert np.array_equal(a, b)
