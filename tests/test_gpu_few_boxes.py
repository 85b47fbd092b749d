"""Products and substitutions of levels with few boxes (bgemv.hip): odd box
sizes and ranks, every number of right-hand sides; a column of a batch equals
its single product bit for bit, whichever launches its sums ran in. And lists
of more terms than are staged at a time."""
import numpy as np
import pytest

import oracle_lib as O
from mxc_amd import _native as N
from mxc_amd.solver import H2, HostLevels, Problem

pytestmark = pytest.mark.gpu


def apply(ctx, call, x):
    n, nr = x.shape
    dx, dy = ctx.array(x), ctx.zeros((n, nr))
    N.check_gpu(call(dx.ptr, dy.ptr, nr, n))
    return dy.download()


@pytest.mark.parametrize("n,leaf,rank", [(40, 20, 7), (131, 65, 33), (520, 65, 20), (3001, 93, 40), (2600, 300, 101)])
@pytest.mark.parametrize("theta", [1.0, 2.0])
def test_batches_equal_single_columns(ctx, n, leaf, rank, theta):
    pts = O.cube_points(n, 41)
    prob = Problem(ctx, pts, leaf)
    A = H2.operator(prob, 1e-10, 0, theta=theta)
    M = H2.preconditioner(prob, rank, 0, theta=theta)
    x = np.random.default_rng(n).uniform(-1, 1, (n, 8))
    gpu, h2 = N.gpu(), N.h2()
    dz = ctx.zeros((n, 8))
    prob.dense_matvec("laplace", 1e3, 0.0, ctx.array(x), dz)
    ref = dz.download()
    dev = h2.mxc_solver_device(A.handle)
    for prec, tol in ((N.MXG_FP64, 1e-8), (N.MXG_FP32, 1e-5)):
        call = lambda p, q, nr, ld: gpu.mxg_h2_matvec(dev, p, q, nr, ld, prec)  # noqa: E731,B023
        one = np.concatenate([apply(ctx, call, x[:, q:q + 1]) for q in range(8)], axis=1)
        # the operator's own tolerance (a hundred of it for the growth over the levels), or FP32's rounding
        assert O.rel_err(one.reshape(-1), ref.reshape(-1)) < tol
        for nr in (2, 3, 5, 8):
            assert np.array_equal(apply(ctx, call, x[:, :nr]), one[:, :nr]), (prec, nr)
    oM = O.Problem(pts, leaf).h2(rank=rank, orth=True, hss_far=True, theta=theta)
    oM.factorize()
    oz = oM.precondition(x[:, 0].copy())
    for prec, tol in ((N.MXG_FP64, 1e-8), (N.MXG_FP32, 1e-3), (N.MXG_BF16, 0.2)):
        assert not M.factorize(prec).any()
        ulv = h2.mxc_solver_ulv(M.handle)

        def call(p, q, nr, ld):
            N.check_gpu(gpu.mxg_memcpy_d2d(ctx.handle, q, p, 8 * nr * ld))
            return gpu.mxg_ulv_solve(ulv, q, nr, ld)  # noqa: B023
        one = np.concatenate([apply(ctx, call, x[:, q:q + 1]) for q in range(8)], axis=1)
        # rounding, or storage, amplified by the conditioning of the rotated blocks
        assert O.rel_err(one[:, 0], oz) < tol, prec
        for nr in (2, 3, 5, 8):
            assert np.array_equal(apply(ctx, call, x[:, :nr]), one[:, :nr]), (prec, nr)


def test_more_terms_than_staged(ctx):
    """1024 boxes of two points, all of them neighbours: 1024 terms per box."""
    n = 2048
    pts = O.cube_points(n, 42)
    prob = Problem(ctx, pts, 2)
    assert prob.levels == 10
    M = H2.preconditioner(prob, 1, 0, theta=1e6)
    x = O.uniform_vec(n, -1, 1, 3)
    dx, dy, dz = ctx.array(x), ctx.zeros(n), ctx.zeros(n)
    M.matvec(dx, dy)  # every block is a near block: the dense product
    prob.dense_matvec("laplace", 1e3, 0.0, dx, dz)
    assert O.rel_err(dy.download(), dz.download()) < 1e-13
    assert not M.factorize(N.MXG_FP64).any()
    M.precondition(dx)
    oM = O.Problem(pts, 2).h2(rank=1, orth=True, hss_far=True, theta=1e6)
    oM.factorize()
    assert O.rel_err(dx.download(), oM.precondition(x)) < 1e-8


@pytest.mark.parametrize("precision,tol", [(N.MXG_FP64, 1e-12), (N.MXG_FP32, 1e-4), (N.MXG_BF16, 1e-1)])
def test_levels_of_empty_boxes(ctx, precision, tol):
    """Leaves of rank 0: the boxes above have no rows. The matrix is its diagonal blocks."""
    n, leaf = 132, 33
    prob = Problem(ctx, O.cube_points(n, 43), leaf)
    assert prob.levels == 2
    rng = np.random.default_rng(4)
    blocks = [rng.uniform(-1, 1, (leaf, leaf)) + 8 * np.eye(leaf) for _ in range(4)]
    alone = [((np.arange(b + 1), np.arange(b)), (np.zeros(b + 1), np.zeros(0))) for b in (1, 2, 4)]
    levels = [dict(dims=[0] * b, ranks=[0] * b, near=near, far=far) for b, (near, far) in zip((1, 2), alone)]
    levels.append(dict(dims=[leaf] * 4, ranks=[0] * 4, near=alone[2][0], far=alone[2][1],
                       A=np.concatenate([b.T.reshape(-1) for b in blocks])))
    M = HostLevels(prob, levels)
    assert not M.factorize(precision).any()
    for nr in (1, 2, 3, 4, 8):
        x = rng.uniform(-1, 1, (n, nr))
        ref = np.concatenate([b @ x[leaf * i:leaf * i + leaf] for i, b in enumerate(blocks)])
        inv = np.concatenate([np.linalg.solve(b, x[leaf * i:leaf * i + leaf]) for i, b in enumerate(blocks)])
        dx, dy = ctx.array(x), ctx.zeros((n, nr))
        M.matvec(dx, dy)
        assert O.rel_err(dy.download().reshape(-1), ref.reshape(-1)) < 1e-13
        M.precondition(dx)  # blocks of condition about 10: rounding, or storage
        assert O.rel_err(dx.download().reshape(-1), inv.reshape(-1)) < tol, nr
    M.close()
