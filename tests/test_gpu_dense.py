"""The matrix-free dense product (kgen.hip) at the edges of its 16-row blocks,
256-column tiles and 8192-column chunks, for every group width, on points that
coincide and for entries that underflow, against numpy in 64 bits."""
import numpy as np
import pytest

import oracle_lib as O
from mxc_amd.solver import Problem

pytestmark = pytest.mark.gpu


def dense(kernel, p, diag, alpha):
    d = np.sqrt(((p[:, None, :] - p[None, :, :]) ** 2).sum(-1))
    with np.errstate(divide="ignore", under="ignore"):
        if kernel == "gaussian":
            return np.where(d == 0, 1.0001, np.exp(-alpha * d * d))
        k = 1.0 / d if kernel == "laplace" else np.exp(-alpha * d) / d
    return np.where(d == 0, diag, k)


@pytest.mark.parametrize("n,nrhs", [(1, 1), (3, 2), (16, 3), (63, 4), (65, 8), (255, 5), (257, 9), (1000, 17), (8193, 1)])
@pytest.mark.parametrize("kernel,alpha", [("laplace", 0.0), ("yukawa", 1.0), ("yukawa", 2000.0), ("gaussian", 3.0),
                                          ("gaussian", 1e5), ("gaussian", -2.0)])
def test_dense_product(ctx, n, nrhs, kernel, alpha):
    pts = O.cube_points(n, 31).reshape(-1, 3)
    pts[n // 2:n // 2 + n // 5] = pts[0]  # coinciding points: off-diagonal entries with the diagonal value
    prob = Problem(ctx, pts.reshape(-1), max(n, 1))
    x = np.random.default_rng(n).uniform(-1, 1, (n, nrhs))
    dx, dy = ctx.array(x), ctx.zeros((n, nrhs))
    prob.dense_matvec(kernel, 1e3, alpha, dx, dy)
    k = dense(kernel, prob.bodies.reshape(-1, 3), 1e3, alpha)
    # an entry to 4 ulp plus the exponential's argument rounded (a relative error
    # of u in alpha d is alpha d u in the entry), and n roundings of the sum
    arg = abs(alpha) * 3 if kernel != "laplace" else 0.0
    bound = (n + 4 + min(arg, 750.0)) * 2.0**-52 * (np.abs(k) @ np.abs(x))
    assert np.all(np.abs(dy.download() - k @ x) <= bound)


@pytest.mark.parametrize("nrhs", [1, 3, 8])
@pytest.mark.parametrize("kernel,alpha", [("laplace", 0.0), ("yukawa", 1.0), ("yukawa", 1e160),
                                          ("gaussian", 1.0), ("gaussian", 1e-308), ("gaussian", 1e300)])
def test_distances_at_the_ends_of_the_number_range(ctx, kernel, alpha, nrhs):
    """Squared distances that overflow, underflow to zero (entries with the
    diagonal value) or to numbers with few bits, and exponents beyond an int."""
    n = 70
    pts = O.cube_points(n, 32).reshape(-1, 3)
    pts[:6] = [[0, 0, 0], [1e-170, 0, 0], [1e-157, 0, 0], [0, 3e-155, 0], [1e155, 0, 0], [0, -2e160, 0]]
    prob = Problem(ctx, pts.reshape(-1), n)
    x = np.random.default_rng(nrhs).uniform(-1, 1, (n, nrhs))
    dx, dy = ctx.array(x), ctx.zeros((n, nrhs))
    prob.dense_matvec(kernel, 1e3, alpha, dx, dy)
    p = prob.bodies.reshape(-1, 3)
    with np.errstate(over="ignore"):
        k = dense(kernel, p, 1e3, alpha)
        d = np.sqrt(((p[:, None, :] - p[None, :, :]) ** 2).sum(-1))
        # an entry to 4 ulp plus its exponent's rounding where it has not underflown, and n roundings of the sum
        arg = np.zeros_like(d) if kernel == "laplace" else alpha * d if kernel == "yukawa" else alpha * d * d
    assert np.isfinite(k).all()
    bound = (n + 4 + np.minimum(arg, 750.0).max()) * 2.0**-52 * (np.abs(k) @ np.abs(x))
    got = dy.download()
    assert np.all(np.abs(got - k @ x) <= bound + 1e-300)
