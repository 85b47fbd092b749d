"""The Householder kernels of the basis construction (qr.hip) at the edges of
their sizes: rows a lane holds (multiples of 64, up to 1024 and beyond),
columns a wave holds, panel widths, full rank and rank one. Two boxes that see
each other: one pivoted QR of an M x M block each."""
import numpy as np
import pytest

import oracle_lib as O
from mxc_amd.solver import H2, Problem
from test_gpu_sketch import first_basis

pytestmark = pytest.mark.gpu

TOL = 1e-4  # truncation: R11's condition number stays near 1 / TOL


def boxes(X, level):
    """Size, rank, Q and R of every box (the oracle's Q and R have the same layout)."""
    dims, ranks = X.dims(level)
    off = np.concatenate([[0], np.cumsum(dims**2)])
    Q, R = X.download(level, 1), X.download(level, 2)
    for i, (m, r) in enumerate(zip(dims, ranks)):
        yield (int(m), int(r), Q[off[i]:off[i + 1]].reshape(m, m, order="F"), R[off[i]:off[i + 1]].reshape(m, m, order="F"))


def compare(X, oX, M, ortho):
    for (m, r, Q, R), (om, orr, oQ, oR) in zip(boxes(X, 1), boxes(oX, 1)):
        assert (m, r) == (om, orr)
        # the same pivots, so Q differs by the rounding of the eliminations (M eps), amplified by R11's conditioning
        tol = 100 * M * 2.0**-52 / TOL
        cols = m if ortho else r
        assert np.abs(Q[:, :cols] - oQ[:, :cols]).max() < tol
        assert np.abs(R[:r, :r] - oR[:r, :r]).max() < tol * max(1, np.abs(oR[:r, :r]).max())
        if ortho and 0 < r < m:
            assert np.abs(Q.T @ Q - np.eye(m)).max() < 10 * m * 2.0**-52


@pytest.mark.parametrize("M,rank", [(2, 1), (40, 24), (64, 64), (65, 33), (129, 110), (192, 8), (200, 128), (257, 100),
                                    (313, 104), (320, 127), (385, 64), (513, 40), (769, 30), (1030, 20)])
def test_orthogonal_bases(ctx, M, rank):
    pts = O.cube_points(2 * M, 11)
    prob, oprob = Problem(ctx, pts, M), O.Problem(pts, M)
    assert prob.levels == 1
    X = H2.preconditioner(prob, rank, 0, eps=TOL)
    oX = oprob.h2(tol=TOL, rank=rank, orth=True, hss_far=True)
    compare(X, oX, M, True)


@pytest.mark.parametrize("M", [2, 63, 129, 256, 313, 520])
def test_interpolative_bases(ctx, M):
    pts = O.cube_points(2 * M, 12)
    prob, oprob = Problem(ctx, pts, M), O.Problem(pts, M)
    X = H2.operator(prob, TOL, 0, theta=0.0)
    oX = oprob.h2(tol=TOL, theta=0.0)
    compare(X, oX, M, False)


@pytest.mark.parametrize("M", [60, 130])
def test_rows_reduced_by_householder(ctx, M):
    """Four boxes, three times as many far rows as columns: the reference's
    row reduction gives the interpolation the sketch gives, to the tolerance."""
    pts = O.cube_points(4 * M, 13)
    prob = Problem(ctx, pts, M)
    x = ctx.array(O.uniform_vec(4 * M, -1, 1, 3))
    y, z = ctx.zeros(4 * M), ctx.zeros(4 * M)
    A = H2.operator(prob, 1e-9, 0, theta=0.0, householder_rows=True)
    A.matvec(x, y)
    prob.dense_matvec("laplace", 1e3, 0.0, x, z)
    # interpolation error: the truncated pivots times a modest growth factor
    assert O.rel_err(y.download(), z.download()) < 1e-9 * 4 * M


@pytest.mark.parametrize("M", [40, 300, 1100])
def test_no_comparable_norm(ctx, M):
    """A far point that is NaN makes every column's norm NaN: the basis shows it (and no column past the last is read)."""
    pts = O.cube_points(2 * M, 14).reshape(-1, 3)
    pts[M + M // 2] = np.nan
    r, q = first_basis(ctx, pts, M, np.arange(M, 2 * M), "laplace")
    assert r > 0 and np.isnan(q).any()
