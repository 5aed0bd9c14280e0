"""The one-launch tail where its forms meet: counts of exactly its LDS room,
captured runs that grow past it and are worked on in place, and more dead slots
than the heads' room holds.  Bit for bit against the launches, which a case of
larger capacity takes."""
import numpy as np
import pytest

from vortex_amd import geometry as geo
from vortex_amd.solver import Case, make_params, VX_PREC_F64, VX_PREC_MIXED

pytestmark = pytest.mark.gpu
VINF = (1.0, 0.0)
ROOM = 3584


def sparse(n, dead, seed):
    """Far enough apart for few merges; `dead` slots without circulation."""
    rng = np.random.default_rng(seed)
    x, y = rng.uniform(1.0, 8.0, n), rng.uniform(-3.0, 3.0, n)
    g = rng.uniform(1e-4, 2e-3, n) * rng.choice([-1.0, 1.0], n)
    g[rng.permutation(n)[:dead]] = 0.0
    return x, y, g


def run(P, state, steps, graph, cap, prec=VX_PREC_F64):
    pan = geo.circle(P, 0.5)
    c = Case(make_params(pan, precision=prec, dt=0.005, r_col_diff_sign=1.0, r_col_same_sign=0.3, n_col=2,
                         ve_size=0.01, max_ve_g=0.02, birth_offset_rel=0.5), pan)
    c.build_matrix()
    c.reserve(cap)
    c.set_state(*state)
    f, counts = c.run_steps_graph(steps, VINF) if graph else (c.run_steps(steps, VINF), None)
    slots = (state[0].size + steps * P + 31) // 32 * 32
    out = (f, *c.state(slots))
    n, caps = c.n, c.capacity
    c.close()
    return n, caps, counts, out


def same(a, b):
    assert a[0] == b[0]
    for p, q in zip(a[3], b[3]):
        assert np.array_equal(p, q)


@pytest.mark.parametrize("prec", [VX_PREC_F64, VX_PREC_MIXED])
@pytest.mark.parametrize("dead", [0, 2200])
def test_growth_past_the_room(dead, prec):
    state = sparse(3400, dead, 5 + dead)
    a, b = run(200, state, 12, True, 0, prec), run(200, state, 12, True, 20000, prec)
    assert a[1] == 8192 and b[1] > 8192
    assert (a[2] > ROOM).sum() >= (6 if dead == 0 else 0) and np.array_equal(a[2], b[2])
    same(a, b)


@pytest.mark.parametrize("n", [ROOM - 65, ROOM - 64, ROOM - 63])
def test_counts_at_the_room(n):
    """64 births make the room's count of slots, one less and one more."""
    state = sparse(n, 0, n)
    a, b = run(64, state, 1, True, 0), run(64, state, 1, True, 20000)
    assert a[1] == 8192
    same(a, b)
    same(run(64, state, 2, False, 0), run(64, state, 2, True, 20000))


@pytest.mark.parametrize("dead", [2047, 2048, 2049, 3000])
def test_more_dead_slots_than_heads(dead):
    state = sparse(3400, dead, dead)
    same(run(64, state, 2, False, 0), run(64, state, 2, True, 20000))
