"""The inverses of the factorization (lu.hip), through a one-box matrix whose
factorization is the inverse of its only block: sizes at the edges of the
16-column panels, of the 64-row tiles and of the workgroup sizes."""
import numpy as np
import pytest

import oracle_lib as O
from mxc_amd import _native as N
from mxc_amd.solver import HostLevels, Problem

pytestmark = pytest.mark.gpu


def solve(ctx, a, b, precision):
    n = len(a)
    prob = Problem(ctx, O.cube_points(n, 3), n)
    assert prob.levels == 0
    none = (np.zeros(2, np.int64), np.zeros(0, np.int64))
    M = HostLevels(prob, [dict(dims=[n], ranks=[0], near=(np.array([0, 1]), np.array([0])), far=none,
                               A=np.asfortranarray(a).reshape(-1, order="F"))])
    info = M.factorize(precision)
    d = ctx.array(b)
    M.precondition(d)
    return d.download(), info


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 63, 64, 65, 96, 192, 213, 256, 257, 511, 512, 513, 1000, 1024])
@pytest.mark.parametrize("precision,u", [(N.MXG_FP64, 2.0**-53), (N.MXG_FP32, 2.0**-24)])
def test_inverse_with_pivoting(ctx, n, precision, u):
    rng = np.random.default_rng(n)
    a = rng.uniform(-1, 1, (n, n))
    a[0, 0] = 0.0 if n > 1 else 0.5  # the first pivot is another row
    x = rng.uniform(-1, 1, n)
    b = a @ x
    y, info = solve(ctx, a, b, precision)
    assert not info.any()
    # an inverse times a vector: n roundings of relative size u per entry of
    # |A^{-1}| |b|, and the elimination's own error of the same form in FP64;
    # for FP32 also the input's and the inverse's rounding
    bound = 4 * (n + 2) * u * np.linalg.cond(a, 2)
    assert O.rel_err(y, x) < bound, (O.rel_err(y, x), bound)


def test_singular_block_is_reported(ctx):
    a = np.ones((40, 40))
    _, info = solve(ctx, a, np.ones(40), N.MXG_FP64)
    assert info.tolist() == [1]
