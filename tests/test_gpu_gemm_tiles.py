"""Batched GEMM at the edges of its tiles: sizes that take each tile height,
ragged last blocks and slabs on either side, with NaN around the operands so
that whatever lies outside them shows when it is used."""
import numpy as np
import pytest

from mxc_amd import _native as N

pytestmark = pytest.mark.gpu


def padded(ctx, a, ld):
    p = np.full((ld, a.shape[1]), np.nan, dtype=a.dtype, order="F")
    p[: a.shape[0]] = a
    return ctx.array(p)


def check(ctx, prec, ta, tb, m, n, k, beta, lda=None):
    dtype = np.float64 if prec == N.MXG_FP64 else np.float32
    rng = np.random.default_rng(m + 3 * n + 7 * k + 2 * ta + tb)
    A = rng.standard_normal((k, m) if ta else (m, k)).astype(dtype)
    B = rng.standard_normal((n, k) if tb else (k, n)).astype(dtype)
    Cm = rng.standard_normal((m, n)).astype(dtype)
    lda, ldb, ldc = lda or A.shape[0] + 3, B.shape[0] + 5, m + 2
    dA, dB, dC = padded(ctx, A, lda), padded(ctx, B, ldb), padded(ctx, Cm, ldc)
    N.check_gpu(N.gpu().mxg_gemm(ctx.handle, prec, ta, tb, m, n, k, -1.5, dA.ptr, lda, dB.ptr, ldb, beta, dC.ptr, ldc))
    got = dC.download()
    assert np.isnan(got[m:]).all()  # nothing written past C's rows
    opA, opB = (A.T if ta else A).astype(np.float64), (B.T if tb else B).astype(np.float64)
    ref = -1.5 * (opA @ opB) + beta * Cm
    scale = 1.5 * (np.abs(opA) @ np.abs(opB)) + abs(beta) * np.abs(Cm)
    # k products and sums, the two scalings and the last sum, each rounded once
    assert (np.abs(got[:m] - ref) <= (k + 4) * np.finfo(dtype).eps * scale + np.finfo(dtype).tiny).all()


@pytest.mark.timeout(120)
@pytest.mark.parametrize("prec", [N.MXG_FP64, N.MXG_FP32])
@pytest.mark.parametrize("m,n", [
    (17, 65), (129, 15),            # one block of F a tile
    (1000, 995),                    # two
    (1490, 1501),                   # four
    (2050, 2033), (113, 33000),     # eight; seven, the F side the rows
    (33000, 97),                    # seven, the F side the columns
])
def test_tile_heights(ctx, prec, m, n):
    for ta, tb, k, beta in ((0, 0, 1, 0.), (0, 1, 17, 0.5), (1, 0, 32, 0.5), (1, 1, 35, 0.)):
        check(ctx, prec, ta, tb, m, n, k, beta)


@pytest.mark.timeout(120)
@pytest.mark.parametrize("prec", [N.MXG_FP64, N.MXG_FP32])
@pytest.mark.parametrize("lda", [(1 << 21) - 1, (1 << 21) + 3])
def test_long_strides(ctx, prec, lda):
    check(ctx, prec, 0, 0, 130, 70, 5, 0.5, lda)
    check(ctx, prec, 1, 0, 66, 70, 18, 0., lda)


@pytest.mark.parametrize("m,n", [(512, 512), (513, 511), (65, 4097), (2047, 2046), (2049, 1985)])  # 64 to 1056 tiles
def test_bf16_tile_orders(ctx, m, n):
    """bfloat16 products of few tiles (runs on an XCD) and of many (launch order), integers: exact."""
    rng = np.random.default_rng(m)
    for ta, tb, k in ((0, 0, 33), (1, 1, 16)):
        A = rng.integers(-8, 9, (k, m) if ta else (m, k)).astype(np.float32)
        B = rng.integers(-8, 9, (n, k) if tb else (k, n)).astype(np.float32)
        Cm = rng.integers(-8, 9, (m, n)).astype(np.float32)
        dA, dB, dC = padded(ctx, A, len(A) + 3), padded(ctx, B, len(B) + 5), padded(ctx, Cm, m + 2)
        N.check_gpu(N.gpu().mxg_gemm(ctx.handle, N.MXG_BF16, ta, tb, m, n, k, 1.0, dA.ptr, len(A) + 3, dB.ptr, len(B) + 5,
                                     2.0, dC.ptr, m + 2))
        got = dC.download()
        assert np.isnan(got[m:]).all()
        assert np.array_equal(got[:m], (A.T if ta else A) @ (B.T if tb else B) + 2 * Cm)
