"""W8A8 and FP8 at up to 64 rows: row counts around a 16-row block, widths on
every workgroup width (one to four 16-column tiles), K around a step, a load
window and the sizes where A no longer fits LDS at once (9216 / 4608 / 2304 k
for 16 / 32 / 64 rows), every form of the kernel that stages A (the choice is
asserted), both sides of the rule between it and the others, and a misaligned
A (the others).

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


# (16-row blocks, column tiles, window, phases) of each shape; None: another
# kernel's
FORMS = [
    (13, 2048, 4000, (1, 1, 8, False)), (13, 4224, 4000, (1, 1, 16, False)), (13, 9984, 4000, (1, 1, 8, True)),
    (16, 1024, 8100, (1, 2, 8, False)), (16, 4096, 8100, (1, 2, 16, False)), (16, 9984, 8100, (1, 2, 16, True)),
    (9, 1024, 8300, (1, 3, 8, False)), (9, 2176, 8300, (1, 3, 16, False)), (9, 9984, 8300, (1, 3, 16, True)),
    (15, 896, 13000, (1, 4, 8, False)), (15, 2176, 13000, (1, 4, 16, False)), (15, 12288, 13000, (1, 4, 16, True)),
    (17, 2048, 4000, (2, 1, 8, False)), (17, 4224, 4000, (2, 1, 16, False)),
    (32, 1024, 8100, (2, 2, 8, False)), (32, 2176, 8100, (2, 2, 16, False)), (32, 5120, 8100, (2, 2, 8, True)),
    (24, 1024, 8300, (2, 3, 8, False)), (24, 2176, 8300, (2, 3, 16, False)), (24, 5120, 8300, (2, 3, 16, True)),
    (29, 896, 13000, (2, 4, 8, False)), (29, 2176, 13000, (2, 4, 16, False)), (29, 5120, 13000, (2, 4, 16, True)),
    (33, 1024, 4000, (4, 1, 8, False)),
    (64, 1024, 8100, (4, 2, 8, False)), (64, 2176, 8100, (4, 2, 16, False)),
    (47, 1024, 8300, (4, 3, 8, False)), (47, 2176, 8300, (4, 3, 16, False)), (47, 2560, 8300, (4, 3, 8, True)),
    (63, 1024, 13000, (4, 4, 8, False)), (63, 2176, 13000, (4, 4, 16, False)), (63, 2560, 13000, (4, 4, 8, True)),
    (2, 2048, 17000, (1, 3, 16, False)), (40, 5120, 17000, (4, 3, 8, True)),  # two rounds of the CUs
    (64, 512, 17000, None), (33, 2048, 17000, None), (1, 4096, 17000, None), (8, 8192, 17000, None),
]


@pytest.mark.parametrize("fp8", [0, 1])
@pytest.mark.parametrize("M,K,N,form", FORMS)
def test_every_form(ops, M, K, N, form, fp8):
    import torch
    f = ops.lib().lhq_selftest_gemm8_stream(M, N, K, fp8)
    assert ((f >> 4 & 15, f & 15, 8 if f & 256 else 16, bool(f & 512)) if f else None) == form
    g = torch.Generator(device="cuda")
    g.manual_seed(M + K + N)
    if not fp8:
        A, B = (torch.randint(-128, 128, s, generator=g, device="cuda", dtype=torch.int8) for s in ((M, K), (K, N)))
        got = ops.gemm_w8a8_i32(A, ops.prepack_b8(B, K, N), M, N, K)
        assert torch.equal(got.long(), (A.double() @ B.double()).long())  # below 2^53: exact
        return
    A, B = ((torch.randn(s, generator=g, device="cuda") * 20).to(torch.float8_e4m3fn) for s in ((M, K), (K, N)))
    C, one = ops.empty((M, N), np.float32), torch.ones(1, device="cuda")
    ops.run("lhq_gemm_fp8_e4m3", A.view(torch.uint8), ops.prepack_b8(B.view(torch.uint8), K, N), one, one, C, M, N, K,
            1.0, 0.0)
    want = A.double() @ B.double()
    assert float((C - want).norm() / want.norm()) <= 1e-4


@pytest.mark.parametrize("lead", [0, 1])
@pytest.mark.parametrize("M,K,N", [(1, 128, 16), (16, 4096, 4100), (24, 4096, 1030), (33, 640, 300), (64, 2432, 700)])
def test_fp8(oracle, ops, M, K, N, lead):
    A = oracle.f32_to_e4m3_n(D.normal((M, K), 20.0, M)).astype(np.uint8)
    B = oracle.f32_to_e4m3_n(D.normal((K, N), 20.0, N)).astype(np.uint8)
    A[M - 1, 5] = 0x7f  # NaN: its row, and no other
    bt = ops.prepack_b8(ops.dev(B), K, N)
    sa, sb = np.array([0.01], np.float32), np.array([0.02], np.float32)
    C0 = D.uniform((M, N), -1, 1, 6)
    C = ops.dev(C0)
    a = ops.dev(np.concatenate([np.zeros(lead, np.uint8), A.ravel()]))[lead:]
    ops.run("lhq_gemm_fp8_e4m3", a, bt, sa, sb, C, M, N, K, 0.5, -1.0)
    got = ops.host(C).astype(np.float64)
    a, b = (oracle.e4m3_to_f32_n(v).astype(np.float64).reshape(v.shape) for v in (A, B))
    with np.errstate(invalid="ignore"):
        want = 0.5 * float(sa[0]) * float(sb[0]) * (a @ b) - C0
    assert np.isnan(got[M - 1]).all() and np.isfinite(got[: M - 1]).all()
    if M > 1:
        assert np.linalg.norm(got[:-1] - want[:-1]) <= 1e-4 * np.linalg.norm(want[:-1])
