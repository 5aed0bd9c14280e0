"""Small counts in fewer launches: the ordered selection as one work-group up
to 8192 items, and the birth right-hand side's expansion sums with one source
per thread.  The compaction that it carries against the oracle's at the edges of
its range; the sums bit for bit against the route with several sources per
thread (the case's empty far tail counted in), and, where the list itself is
long, by adding up two halves."""
import numpy as np
import pytest

from vortex_amd import geometry as geo
from vortex_amd.solver import Case, make_params, VX_PREC_F64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 1023, 1024, 1025, 4096, 8160, 8191, 8192, 8193, 12345])
@pytest.mark.parametrize("dead", [0.0, 0.3, 0.97, 1.0])
def test_selection(ref, n, dead):
    rng = np.random.default_rng(n)
    x, y, g = rng.uniform(1, 2, n), rng.uniform(1, 2, n), rng.uniform(0.1, 1.0, n)
    g[rng.random(n) < dead] = 0.0
    pan = geo.circle(8, 0.5)
    c = Case(make_params(pan, precision=VX_PREC_F64), pan)
    c.set_state(x, y, g)
    c.compact()
    xr, yr, gr, nr = ref.compact(x, y, g)
    assert c.n == nr
    for a, b in zip(c.state(n), (xr, yr, gr)):
        assert np.array_equal(a, b)
    c.close()


def cloud(n, near):
    rng = np.random.default_rng(n + near)
    r, a = rng.uniform(0.501, 0.99 if near else 6.0, n), rng.uniform(0.0, 2 * np.pi, n)
    return r * np.cos(a), r * np.sin(a), rng.uniform(-1.0, 1.0, n)


@pytest.mark.parametrize("near", [0, 1])
@pytest.mark.parametrize("n", [1, 255, 256, 257, 8191, 8192])
def test_one_source_per_thread(n, near):
    pan = geo.circle(200, 0.5)
    c = Case(make_params(pan, precision=VX_PREC_F64), pan)
    c.reserve(131104)
    c.set_state(*cloud(n, near))
    few, many = c.right_part(n, (1.0, 0.2)), c.right_part(131104, (1.0, 0.2))
    c.close()
    assert np.all(np.isfinite(few)) and np.array_equal(few, many)


def test_long_list_adds_up():
    """9001 listed sources (several per thread) against halves of 4500 and 4501:
    each sum's rounding is below n eps of its terms' size, sum |g| / (2 pi d)
    with d the smallest distance; the truncation of the expansions is 2^-47 of
    the same."""
    pan, n = geo.circle(200, 0.5), 9001
    x, y, g = cloud(n, 1)
    c = Case(make_params(pan, precision=VX_PREC_F64), pan)

    def rhs(s):
        c.set_state(x[s], y[s], g[s])
        return c.right_part(x[s].size, (0.0, 0.0))

    whole, halves = rhs(slice(0, n)), rhs(slice(0, 4500)) + rhs(slice(4500, n))
    c.close()
    tol = (2 * n * np.finfo(float).eps + 2.0 ** -46) * np.abs(g).sum() / (2 * np.pi * 0.001)
    assert np.all(np.isfinite(whole)) and np.max(np.abs(whole - halves)) <= tol
