"""Device-count steps of a case whose capacity lies far above its count: the
direct kernels' partial sums take the memory that some count up to the capacity
needs, not the product of the largest counts and the most runs, and the bounded
grids cover every count at every number of targets per thread."""
import numpy as np
import pytest
import torch

from vortex_amd import geometry as geo
from vortex_amd.solver import Case, make_params, VX_PREC_F64, VX_PREC_MIXED
from vortex_amd.state import uniform_wake

pytestmark = pytest.mark.gpu
VINF = (1.0, 0.0)


def case(prec, cap):
    pan = geo.circle(64, 0.5)
    c = Case(make_params(pan, precision=prec, dt=0.005, nu=1e-3, r_col_diff_sign=0.3, r_col_same_sign=0.3,
                         birth_offset_rel=0.5), pan)
    c.build_matrix()
    c.reserve(cap)
    return c


@pytest.mark.parametrize("prec", [VX_PREC_F64, VX_PREC_MIXED])
def test_graph_workspace_follows_the_need(prec):
    """Capacity 400000: six doubles for 400000 + 2^20 targets and runs are 70 MB
    (an eighth to spare on top); every other buffer of a case is linear in the
    capacity, below 500 bytes a slot in all (200 MB)."""
    c = case(prec, 400000)
    c.set_state(*uniform_wake(300, seed=1))
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    c.run_steps_graph(2, VINF)
    used = free - torch.cuda.mem_get_info()[0]
    c.close()
    print(f"[graph] prec={prec} workspace {used / 1e6:.0f} MB", flush=True)
    assert used < 300e6


@pytest.mark.parametrize("prec,tpt", [(VX_PREC_F64, 0), (VX_PREC_F64, 8), (VX_PREC_MIXED, 0), (VX_PREC_MIXED, 2),
                                      (VX_PREC_MIXED, 8)])
@pytest.mark.parametrize("n", [300, 16200, 16500, 40000])
def test_graph_far_below_its_capacity_equals_stream_steps(prec, tpt, n):
    out = []
    for graph in (False, True):
        c = case(prec, 1000000 if graph else 0)
        c.set_tuning(tpt_bs=tpt, tpt_diff=tpt)
        c.set_state(*uniform_wake(n, seed=4, max_ve_g=1e-4))
        f = c.run_steps_graph(4, VINF)[0] if graph else c.run_steps(4, VINF)
        out.append((c.n, f, *c.state()))
        c.close()
    assert out[0][0] == out[1][0]
    for a, b in zip(out[0][1:], out[1][1:]):
        assert np.array_equal(a, b)
