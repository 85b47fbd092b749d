"""GMRES at the edges of its reductions: vectors of one block of rows and a
little more or less, more blocks than a wave has lanes, and a restart whose
least-squares problem does not fit LDS."""
import numpy as np
import pytest

import oracle_lib as O
from mxc_amd import _native as N
from mxc_amd.solver import H2, Problem

pytestmark = pytest.mark.gpu


@pytest.mark.timeout(120)
@pytest.mark.parametrize("n,restart", [(255, 10), (256, 10), (257, 10), (4097, 10), (16640, 10), (257, 100)])
@pytest.mark.parametrize("mode", [N.GMRES_REFERENCE, N.GMRES_CGS2])
def test_residual_is_the_solution_s(ctx, n, restart, mode):
    prob = Problem(ctx, O.cube_points(n, 3), 128)
    A, M = H2.operator(prob, 1e-10, 500), H2.preconditioner(prob, 60, 500)
    M.factorize(N.MXG_FP64)
    b = O.uniform_vec(n, -1, 1, 9)
    db, dx, dy = ctx.array(b), ctx.zeros(n), ctx.zeros(n)
    resid, iters, inner = A.gmres(M, db, dx, 1e-10, restart=restart, max_cycles=20, mode=mode)
    assert resid[-1] < 1e-10
    A.matvec(dx, dy)
    # two FP64 products of x: each within a few hundred roundings of |A| |x| ~ |b|
    assert abs(np.linalg.norm(b - dy.download()) / np.linalg.norm(b) - resid[-1]) < 1e-13
    M.close()
    A.close()
    prob.close()
