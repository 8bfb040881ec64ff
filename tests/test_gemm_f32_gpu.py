"""fp32 GEMM tiles at their edges: rows and columns around a tile, K around the
32-deep stage and below one stage per wave, misaligned operands, each launch
shape, the VALU tiles of short K beside them, denormals, Inf and NaN, against
numpy in 64 bits.

Tolerance: every output is a sum of K rounded products in some order, so its
error is at most K * 2^-24 * sum |a b| (any order, fp32, unit roundoff 2^-24),
plus two roundings of the epilogue.
"""
import numpy as np
import pytest

from tests import _data as D

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops(lib):
    from longhornai_amd import ops as _ops
    return _ops


def _check(got, A, B, C0, alpha, beta):
    K = A.shape[-1]
    A, B, C0 = (v.astype(np.float64) for v in (A, B, C0))
    want = alpha * (A @ B) + beta * C0
    bound = 2.0 ** -24 * ((K + 2) * abs(alpha) * (np.abs(A) @ np.abs(B)) + 3 * np.abs(beta * C0) + 2 * np.abs(want))
    assert (np.abs(got - want) <= bound).all()


# 64x32 tiles on 4 waves from 1024 tiles, on 8 from 256, 32x32 below; the last
# three rows are VALU tiles but for their first shape (K, rows and outputs on
# both sides of that line)
@pytest.mark.parametrize("M,K,N", [
    (1, 1, 1), (31, 31, 33), (33, 32, 32), (32, 33, 31), (5, 7, 300), (40, 255, 65), (1, 289, 1000),
    (65, 100, 4097), (128, 96, 4095), (129, 70, 4100),
    (1024, 260, 2049), (4097, 300, 500), (2049, 257, 1030),
    (33, 23, 600), (1, 23, 600), (300, 23, 1000), (512, 31, 1025), (512, 63, 1025), (17, 32, 16500),
    (1090, 95, 1025), (1024, 67, 2049), (4097, 40, 500), (65, 16, 4097), (4, 33, 8192), (4, 33, 8193),
])
@pytest.mark.parametrize("lead", [0, 1])
def test_shapes(ops, M, K, N, lead):
    A, B, C0 = D.normal((M, K), 1.0, M), D.normal((K, N), 1.0, N), D.normal((M, N), 1.0, K)
    def off(a):
        return ops.dev(np.concatenate([np.zeros(lead, np.float32), a.ravel()]))[lead:]
    for fn, alpha, beta in (("lhq_gemm_f32", 1.0, 0.0), ("lhq_gemm_f32", 0.5, 1.0), ("lhq_gemm_f32_ref", -1.5, 0.25)):
        C = off(C0)
        ops.run(fn, off(A), off(B), C, M, N, K, alpha, beta)
        _check(ops.host(C).reshape(M, N), A, B, C0, alpha, beta)


@pytest.mark.parametrize("batch,M,K,N", [(300, 33, 65, 34), (60, 33, 65, 34), (60, 65, 257, 290), (9, 65, 257, 8200)])
def test_batched(ops, batch, M, K, N):
    A, B = D.normal((batch, M, K), 1.0, 1), D.normal((batch, K, N), 1.0, 2)
    C0 = D.normal((batch, M, N), 1.0, 3)
    C = ops.dev(C0)
    ops.run("lhq_gemm_f32_batched", A, B, C, batch, M, N, K, 2.0, -1.0)
    _check(ops.host(C), A, B, C0, 2.0, -1.0)


def test_empty_sum_and_unread_output(ops):
    C = ops.dev(np.full((3, 5), np.nan, np.float32))
    ops.run("lhq_gemm_f32", None, None, C, 3, 5, 0, 1.0, 0.0)
    assert (ops.host(C) == 0).all()
    # one shape for each tile: VALU, 64 x 32 on 4 and 8 waves, 32 x 32 on 8
    for M, K, N in ((517, 2, 1), (2048, 96, 1024), (100, 257, 4096), (33, 70, 40)):
        C = ops.dev(np.full((M, N), np.nan, np.float32))
        ops.run("lhq_gemm_f32", np.ones((M, K), np.float32), np.ones((K, N), np.float32), C, M, N, K, 1.0, 0.0)
        assert (ops.host(C) == K).all(), (M, K, N)


def test_more_rows_than_the_valu_grid_holds(ops):
    M = 64 * 65535 + 1
    A = (np.arange(2 * M, dtype=np.int64) % 1021).astype(np.float32).reshape(M, 2)
    C = ops.empty((M, 1), np.float32)
    ops.run("lhq_gemm_f32", A, np.array([[1.0], [2.0]], np.float32), C, M, 1, 2, 1.0, 0.0)
    assert np.array_equal(ops.host(C)[:, 0], A[:, 0] + 2 * A[:, 1])  # whole numbers: exact


def test_denormals_and_non_finite(ops):
    M, K, N = 40, 70, 40
    A, B = np.full((M, K), 1e-30, np.float32), np.full((K, N), 1e-12, np.float32)
    C = ops.empty((M, N), np.float32)
    ops.run("lhq_gemm_f32", A, B, C, M, N, K, 1.0, 0.0)
    # each denormal product is within half a step (2^-150) and so is each sum
    assert np.abs(ops.host(C).astype(np.float64) - K * 1e-42).max() <= 2 * K * 2.0 ** -150
    A, B = D.normal((M, K), 1.0, 4), D.normal((K, N), 1.0, 5)
    A[3, 69], A[7, 2], B[69, 5] = np.inf, np.nan, -np.inf
    ops.run("lhq_gemm_f32", A, B, C, M, N, K, 1.0, 0.0)
    with np.errstate(invalid="ignore"):
        want = A.astype(np.float64) @ B.astype(np.float64)
    got = ops.host(C)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
