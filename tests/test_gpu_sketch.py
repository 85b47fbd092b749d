"""The far-field sketch (sketch.hip) at the edges of its tiles, slices and
scaling: ranks and interpolative bases against the oracle's FP64 sketch of the
same blocks, and the product against the dense one."""
import numpy as np
import pytest

import oracle_lib as O
from mxc_amd.solver import H2, Problem

pytestmark = pytest.mark.gpu

TOL = 1e-5


def check(ctx, pts, leaf, kernel="laplace", alpha=1.0, tol=TOL, same_bases=True):
    prob, oprob = Problem(ctx, pts, leaf), O.Problem(pts, leaf)
    n, L = prob.n, prob.levels
    A = H2.operator(prob, tol, 0, kernel, 1e3, alpha, 0.0)  # theta 0: every other box is far
    oA = oprob.h2(kernel=kernel, alpha=alpha, theta=0.0, tol=tol)
    dims, ranks = A.dims(L)
    assert np.array_equal(ranks, oA.dims(L)[1])
    if same_bases:
        # the same pivots; the interpolation's rounding error is amplified by
        # the condition number of the kept columns, about 1 / tol
        q, oq = A.download(L, 1), oA.download(L, 1)
        assert np.abs(q - oq).max() < 100 * dims.max() * 2.0**-52 / tol
    x = O.uniform_vec(n, -1, 1, 5)
    dx, dy, dz = ctx.array(x), ctx.zeros(n), ctx.zeros(n)
    A.matvec(dx, dy)
    prob.dense_matvec(kernel, 1e3, alpha, dx, dz)
    # truncated pivots, the growth of the interpolation and the levels
    assert O.rel_err(dy.download(), dz.download()) < 100 * tol


@pytest.mark.parametrize("M", [17, 64, 65, 128, 129, 256, 257, 384, 385, 512, 530])
@pytest.mark.parametrize("kernel", ["laplace", "yukawa"])
def test_tile_shapes(ctx, M, kernel):
    check(ctx, O.cube_points(4 * M, 21), M, kernel)


@pytest.mark.parametrize("n,leaf", [(9700, 303), (8192 + 64, 64)])  # more than one slice; a slice of few rows
def test_slices(ctx, n, leaf):
    check(ctx, O.cube_points(n, 22), leaf)


@pytest.mark.parametrize("kernel,alpha", [("gaussian", 1.0), ("gaussian", 300.0), ("yukawa", 40.0), ("yukawa", -2.0),
                                          ("gaussian", -1.0)])
def test_range_of_the_entries(ctx, kernel, alpha):
    """Entries over many orders of magnitude, and kernels that grow with the distance."""
    check(ctx, O.cube_points(1500, 23), 187, kernel, alpha, same_bases=False)


def test_coinciding_points(ctx):
    """Copies of a point in several boxes: far entries with the diagonal value."""
    pts = O.cube_points(1200, 24).reshape(-1, 3)
    pts[300:900] = pts[0]
    check(ctx, pts.reshape(-1), 150, same_bases=False)
