"""The far-field sketch (sketch.hip) at the edges of its tiles, slices and
scaling: ranks and interpolative bases against the oracle's FP64 sketch of the
same blocks, and the product against the dense one."""
import ctypes as C

import numpy as np
import pytest
import scipy.linalg

import oracle_lib as O
from mxc_amd import _native as N
from mxc_amd.device import kernel_desc
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


def first_basis(ctx, pts, M, far, kernel, diag=1e3, alpha=1.0):
    """Rank and interpolative basis (M x M) of the box of the first M points for an explicit far list."""
    G, n = N.gpu(), len(pts)
    i64 = lambda *a: np.array(a, np.int64)  # noqa: E731
    pts, far = np.ascontiguousarray(pts), np.asarray(far, np.int64)
    dims, begin, rp, col, none = i64(M, n - M), i64(0, M), i64(0, 2, 4), i64(0, 1, 0, 1), i64(0, 0, 0)
    off, ranks = i64(0, len(far), len(far)), i64(0, 0)
    h = C.c_void_p()
    N.check_gpu(G.mxg_h2_create(ctx.handle, kernel_desc(kernel, diag, alpha), pts.ctypes.data, n, 1, 0, C.byref(h)))
    N.check_gpu(G.mxg_h2_construct_level(h, 1, 2, *(a.ctypes.data for a in (dims, begin, rp, col, none, none, off, far)),
                                         1e-2, 0, 0, ranks.ctypes.data))
    q = np.zeros(G.mxg_h2_level_size(h, 1, N.H2_BASIS))
    N.check_gpu(G.mxg_h2_download(h, 1, N.H2_BASIS, q.ctypes.data, len(q)))
    G.mxg_h2_destroy(h)
    return ranks[0], q[:M * M].reshape(M, M).T


def apart(M, rows, seed):
    """M points in a cube of side 0.2 amid rows outside of a cube of side 0.4, the first row but one in its middle."""
    p = O.cube_points(M + 2 * rows, seed).reshape(-1, 3)
    cols, others = 0.4 + 0.2 * p[:M], p[M:]
    others = others[np.abs(others - 0.5).max(1) > 0.2][:rows]
    others[1] = [0.5, 0.503, 0.5]
    return np.concatenate([cols, others])


@pytest.mark.parametrize("M", [40, 300])
@pytest.mark.parametrize("kernel,away", [("laplace", [1e155, 1e160]), ("yukawa", [1e12, 1e155, 1e160]),
                                         ("gaussian", [1e7, 1e155, 1e160])])
def test_far_rows_with_zero_entries(ctx, M, kernel, away):
    """Rows whose squared distance overflows, or whose exponential is zero, add nothing."""
    pts = apart(M, 700 + len(away), 25)
    pts[M + 700:] = np.array(away)[:, None] * [1.0, -0.5, 0.25]
    far = np.arange(M, len(pts))
    r, q = first_basis(ctx, pts, M, far, kernel)
    r0, q0 = first_basis(ctx, pts, M, far[:700], kernel)
    assert 0 < r0 < M and np.isfinite(q0).all()
    assert r == r0 and np.array_equal(q, q0)


@pytest.mark.parametrize("M", [40, 300])
@pytest.mark.parametrize("kernel", ["laplace", "yukawa", "gaussian"])
def test_distances_that_underflow(ctx, M, kernel):
    """A far row at a distance whose square is zero has the diagonal value, as if it coincided."""
    pts = apart(M, 700, 26) - 0.5
    pts[3] = pts[M + 5] = 0.0
    r0, q0 = first_basis(ctx, pts, M, np.arange(M, len(pts)), kernel)
    pts[M + 5] = [1e-170, 0.0, 0.0]
    r, q = first_basis(ctx, pts, M, np.arange(M, len(pts)), kernel)
    assert 0 < r0 < M and r == r0 and np.array_equal(q, q0)


@pytest.mark.parametrize("M", [40, 300])
@pytest.mark.parametrize("case", ["diagonal", "column", "overflow"])
def test_columns_that_are_not_finite(ctx, M, case):
    """Entries that are not finite spoil their own columns, visibly: a diagonal value that is NaN with coinciding
    points, a column point that is NaN, a kernel that overflows for one pair. The others' bases are as ever."""
    pts = apart(M, 700, 27)
    col, diag, kernel, alpha = 3, 1e3, "laplace", 1.0
    far = np.arange(M, len(pts))
    if case == "diagonal":
        pts[M + 9], diag = pts[col], np.nan
    elif case == "column":
        pts[col] = np.nan
    else:
        kernel, alpha = "gaussian", -200.0  # columns of squares that are still finite
        pts[M + 10] = [10.0, 0.5, 0.5]
        far = far[far != M + 10]
        pts[col] = [9.5, 0.5, 0.5]  # 9 from the other columns' middle: exp(200 81) against every row
    r, q = first_basis(ctx, pts, M, far, kernel, diag, alpha)
    assert 0 < r < M
    rest = np.arange(M) != col
    assert np.isnan(q[col, :r]).all() and np.isfinite(q[rest]).all()
    # the same with a column of zeros in its place, or for a kernel without any, of NaN
    pts[col] = np.nan if case == "overflow" else 1e160
    r0, q0 = first_basis(ctx, pts, M, far, kernel, 1e3, alpha)
    assert r == r0 and np.abs(q[rest] - q0[rest]).max() < 1e-9


def signs(t, i):
    """The sketch's sign of far row t and row i: bit i % 64 of a 64-bit hash of (t, i / 64)."""
    with np.errstate(over="ignore"):
        z = (t[None, :] * np.uint64(0x9E3779B97F4A7C15) + (i >> np.uint64(6))[:, None] * np.uint64(0xD1B54A32D192ED03)
             + np.uint64(0x632BE59BD9B4E019))
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        z ^= z >> np.uint64(31)
    return 1.0 - 2.0 * ((z >> (i & np.uint64(63))[:, None]) & np.uint64(1)).astype(np.float64)


@pytest.mark.parametrize("M,nf", [(40, 131072 - 70), (40, 131072 + 70), (70, 2 * 131072 + 8192 + 1), (1030, 5 * 8192 + 3)])
def test_long_far_lists(ctx, M, nf):
    """Lists of more far rows than the table of signs holds at a time, against the same sketch in numpy."""
    rows = 900
    pts = apart(M, rows, 28)
    far = M + np.arange(nf) * 7 % rows  # every row again and again
    r, q = first_basis(ctx, pts, M, far, "laplace")
    per_row = np.zeros((M, rows))  # the signs of each body's rows, summed
    for a in range(0, nf, 8192):
        t = np.arange(a, min(a + 8192, nf))
        s = signs(t.astype(np.uint64), np.arange(M, dtype=np.uint64))
        for b in range(rows):
            per_row[:, b] += s[:, far[t] - M == b].sum(1)
    G = 1.0 / np.sqrt(((pts[M:, None, :] - pts[None, :M, :]) ** 2).sum(-1))
    _, R, piv = scipy.linalg.qr(per_row @ G, mode="economic", pivoting=True)
    d = np.abs(np.diag(R))
    k = int((d > 1e-2 * d.max()).sum())
    assert 0 < k < M and r == k
    ref = np.zeros((M, k))
    ref[piv[:k]] = np.eye(k)
    ref[piv[k:]] = np.linalg.solve(R[:k, :k], R[:k, k:]).T
    # the same pivots: rounding, amplified by the conditioning of the kept columns, about 100
    assert np.abs(q[:, :k] - ref).max() < 1e4 * M * 2.0**-52


def test_memory_of_long_far_lists(ctx):
    """The table of signs stays small beside the list itself."""
    hip = C.CDLL("libamdhip64.so")

    def free():
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value
    M, rows, nf = 40, 900, 4 << 20
    pts = apart(M, rows, 29)
    first_basis(ctx, pts, M, M + np.arange(9000) % rows, "laplace")
    before = free()
    first_basis(ctx, pts, M, M + np.arange(nf) % rows, "laplace")
    # the list (4 bytes an entry), the table (64 MB) and slices, all kept by the context's pool at most
    assert before - free() < 4 * nf + (96 << 20)
