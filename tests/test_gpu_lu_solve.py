"""Refined solves around the block edges: the stopping test's bound holds for
the residual taken in FP64 on the host, a zero right-hand side needs no
correction, and solves in a row do not disturb each other (the counters that
they share)."""
import numpy as np
import pytest

from vortex_amd import geometry as geo
from vortex_amd.solver import Case, make_params, VX_FLAG_LU_REFINE, VX_PREC_MIXED

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("P", [3, 62, 63, 64, 65, 255, 511, 512, 1023])
def test_solve(P):
    pan = geo.circle(P, 0.5)
    c = Case(make_params(pan, precision=VX_PREC_MIXED, flags=VX_FLAG_LU_REFINE), pan)
    c.build_matrix()
    A, n = c.panel_matrix(), P + 1
    rng = np.random.default_rng(P)
    seen = {}
    for k in (0, 1, 2, 0, 1):
        R, d_g = (np.zeros(P), 0.0) if k == 2 else (rng.uniform(-1.0, 1.0, P) if k not in seen else seen[k][0], 0.25 * k)
        c.n = 0
        x = c.birth(R, d_g)
        info = c.solve_info()
        assert info["converged"] and info["iters"] == 0 if k == 2 else info["converged"] and info["iters"] > 0
        if k == 2:
            assert not np.any(x)
        elif k in seen:
            assert np.array_equal(x, seen[k][1])
        seen[k] = (R, x)
        # ||b - A x|| <= ||A|| ||x|| eps sqrt(n), and the host's own rounding, n eps of the
        # same; x holds all unknowns but the last, which the last panel row's test cannot see
        r = (R - A[:P, :P] @ x)
        lam = np.dot(r, A[:P, P]) / np.dot(A[:P, P], A[:P, P])
        norm_a, norm_x = np.abs(A).sum(1).max(), max(np.abs(x).max(), abs(lam))
        bound = (np.sqrt(n) + n) * np.finfo(float).eps * norm_a * norm_x
        assert np.abs(r - lam * A[:P, P]).max() <= 2 * bound  # lam itself carries the residual once more
    c.close()
