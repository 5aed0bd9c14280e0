"""Blocked Gauss-Jordan inverse of the panel system (vx_case_build_matrix) at
the edges of its blocks and of its panel shapes (rows per thread change at
256, 512, 1024, 2048, 3072 and 4096 rows).

Tolerances: against the oracle's inverse 1e-10 of the largest entry, as
elsewhere; the residual |M L - I| at most 64 m u |M|_inf |L|_inf, elimination
with partial pivoting being backward stable up to its pivot growth."""
import numpy as np
import pytest

from vortex_amd import geometry as geo
from vortex_amd._lib import VortexError
from vortex_amd.solver import Case, make_params, VX_PREC_F64

pytestmark = pytest.mark.gpu


def build(pan):
    c = Case(make_params(pan, precision=VX_PREC_F64), pan)
    c.build_matrix()
    L, M = c.panel_matrix(), c.matrix()
    c.close()
    return L, M


@pytest.mark.parametrize("P", [4, 15, 16, 17, 31, 255, 256, 257, 511, 513])
@pytest.mark.parametrize("maker", [geo.circle, lambda P: geo.flat_plate(P, alpha_deg=9.0)])
def test_inverse_small(ref, maker, P):
    L, M = build(maker(P))
    Mr = ref.invert(L, 1)
    assert np.max(np.abs(M - Mr)) <= 1e-10 * np.max(np.abs(Mr))


@pytest.mark.parametrize("P", [1023, 1024, 1030, 2047, 2048, 3071, 3073, 4097])
def test_inverse_residual(P):
    L, M = build(geo.flat_plate(P, alpha_deg=9.0))
    norm = lambda A: np.max(np.sum(np.abs(A), axis=1))  # noqa: E731
    R = M @ L - np.eye(P + 1)
    assert np.max(np.abs(R)) <= 64 * (P + 1) * 2.0 ** -53 * norm(M) * norm(L)


def test_singular_system_is_an_error():
    pan = geo.circle(40)
    pan[7] = pan[6]  # two panels in one place
    c = Case(make_params(geo.circle(40), precision=VX_PREC_F64), pan)
    with pytest.raises(VortexError):
        c.build_matrix()
    c.close()
