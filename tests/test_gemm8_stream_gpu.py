"""W8A8 and FP8 at up to 64 rows: row counts around a 16-row block, widths on
every workgroup width (one to four 16-column tiles), K around a step, a load
window and the sizes where A no longer fits LDS at once (9216 / 4608 / 2304 k
for 16 / 32 / 64 rows), and a misaligned A (the other kernel).

int8: the int32 accumulators exactly, and the fp32 and bf16 outputs bit for
bit against the oracle.  fp8: sums inside the matrix instruction are not those
of fp32, so the bar of the fp8 tests, 1e-4 relative Frobenius.
"""
import numpy as np
import pytest

from tests import _data as D

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops(lib):
    from longhornai_amd import ops as _ops
    return _ops


def _i8(shape, seed):
    return D.rng(seed).integers(-128, 128, shape).astype(np.int8)


SHAPES = [
    (1, 16, 1), (2, 64, 17), (15, 80, 300), (16, 1040, 47), (17, 4096, 4100), (31, 512, 14336), (32, 528, 10240),
    (33, 576, 33), (63, 1024, 4097), (64, 2304, 700), (64, 2320, 8200), (48, 4096, 14336), (65, 512, 300),
    (16, 9216, 500), (16, 9232, 500), (9, 10000, 12300), (32, 4608, 800), (32, 4624, 800), (20, 12304, 10240),
]


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("lead", [0, 1])
def test_int8_exact(ops, M, K, N, lead):
    A, B = _i8((M, K), M + K), _i8((K, N), N)
    bt = ops.prepack_b8(ops.dev(B), K, N)
    a = ops.dev(np.concatenate([np.zeros(lead, np.int8), A.ravel()]))[lead:]
    C = ops.dev(np.full((M, N), 7, np.int32))
    got = ops.host(ops.gemm_w8a8_i32(a, bt, M, N, K, C))
    want = A.astype(np.float64) @ B.astype(np.float64)  # below 2^53: exact
    assert np.array_equal(got, want.astype(np.int64))


@pytest.mark.parametrize("M,K,N", [(17, 512, 300), (64, 2320, 130), (3, 96, 50)])
def test_int8_epilogues(oracle, ops, M, K, N):
    A, B = _i8((M, K), 1), _i8((K, N), 2)
    As, Bs, C0 = D.uniform((M,), 0.01, 1, 3), D.uniform((N,), 0.01, 1, 4), D.uniform((M, N), -9, 9, 5)
    bt = ops.prepack_b8(ops.dev(B), K, N)
    for alpha, beta in ((1.0, 0.0), (0.5, 1.0), (-1.5, 0.25)):
        C = ops.dev(C0)
        ops.run("lhq_gemm_w8a8", A, bt, As, Bs, C, M, N, K, alpha, beta)
        assert ops.host(C).tobytes() == oracle.gemm_w8a8(A, B, As, Bs, C0, alpha, beta).tobytes()
    got = ops.host(ops.gemm_w8a8_bf16(ops.dev(A), bt, ops.dev(As), ops.dev(Bs), M, N, K), np.uint16)
    assert got.tobytes() == oracle.gemm_w8a8_bf16out(A, B, As, Bs).tobytes()


@pytest.mark.parametrize("M,K,N", [(1, 128, 16), (16, 4096, 4100), (24, 4096, 1030), (33, 640, 300), (64, 2432, 700)])
def test_fp8(oracle, ops, M, K, N):
    A = oracle.f32_to_e4m3_n(D.normal((M, K), 20.0, M)).astype(np.uint8)
    B = oracle.f32_to_e4m3_n(D.normal((K, N), 20.0, N)).astype(np.uint8)
    A[M - 1, 5] = 0x7f  # NaN: its row, and no other
    bt = ops.prepack_b8(ops.dev(B), K, N)
    sa, sb = np.array([0.01], np.float32), np.array([0.02], np.float32)
    C0 = D.uniform((M, N), -1, 1, 6)
    C = ops.dev(C0)
    ops.run("lhq_gemm_fp8_e4m3", A, bt, sa, sb, C, M, N, K, 0.5, -1.0)
    got = ops.host(C).astype(np.float64)
    a, b = (oracle.e4m3_to_f32_n(v).astype(np.float64).reshape(v.shape) for v in (A, B))
    with np.errstate(invalid="ignore"):
        want = 0.5 * float(sa[0]) * float(sb[0]) * (a @ b) - C0
    assert np.isnan(got[M - 1]).all() and np.isfinite(got[: M - 1]).all()
    if M > 1:
        assert np.linalg.norm(got[:-1] - want[:-1]) <= 1e-4 * np.linalg.norm(want[:-1])
