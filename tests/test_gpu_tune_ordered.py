"""Autotuning where the direct kernels do not use the targets per thread (FP64, at
most 16384 sources): whichever was the luckiest must not be carried on to counts
that do."""
import pytest

from vortex_amd import geometry as geo
from vortex_amd.solver import Case, make_params, VX_PREC_F64
from vortex_amd.state import uniform_wake

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [500, 16384])
@pytest.mark.parametrize("bs,diff", [(0, 0), (2, 4)])
def test_setting_stays(n, bs, diff):
    pan = geo.circle(64, 0.5)
    c = Case(make_params(pan, precision=VX_PREC_F64, ve_size=0.004), pan)
    c.set_state(*uniform_wake(n, seed=5))
    c.set_tuning(tpt_bs=bs, tpt_diff=diff)
    t = c.autotune((1.0, 0.0))
    kept = c.tuning()
    c.close()
    assert (t["tpt_bs"], t["tpt_diff"]) == (kept["tpt_bs"], kept["tpt_diff"]) == (bs, diff)
    assert t["trials"] == 2 and 0 < t["ms_best"] == t["ms_default"]
