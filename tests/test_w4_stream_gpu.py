"""The W4A16 kernel for a few rows (weights streamed, rows staged in LDS; the
workspace and no-allocation entry points and the fp32 interface take it by a
rule) and the calls on both sides of that rule: 5 to 64 rows with ragged row
blocks, one column tile to two rounds of the CUs, one K tile, K phases that end
mid-window, G = 32 to 384, zero points, alpha / beta.  Every form of the kernel
that the rule can choose is run, and the choice asserted.

Tolerance, against float64 on the same codes: the terms are x (144 + u - z) and
-144 x, so a partial sum never exceeds 303 sum_k s |x|, and each of the at most
2 K + 2 K/G + 8 additions (twice for fp32, hi and lo planes) rounds once
(2^-24); plus half an ulp of the result: 2^-8 |want| in bf16, 2^-24 in fp32,
whose hi + lo planes hold each activation to 2^-17.
"""
import numpy as np
import pytest

from tests import _data as D

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops(lib):
    from longhornai_amd import ops as _ops
    return _ops


def _codes(K, N, G, seed):
    g = D.rng(seed)
    u = g.integers(0, 16, (K, N)).astype(np.uint8)
    z = g.integers(0, 16, (K // G, N)).astype(np.uint8)
    s = (0.01 * np.exp(0.3 * g.standard_normal((K // G, N)))).astype(np.float16)
    return u, z, s, (u[0::2] | (u[1::2] << 4)).astype(np.uint8)


def _form(ops, M, N, K, G, f32=0):
    """(16-row blocks, column tiles per workgroup) of the kernel, or None."""
    f = ops.lib().lhq_selftest_w4_stream(M, N, K, G, f32)
    return divmod(f, 16) if f else None


def _bf16_call(ops, entry, A, w):
    M = A.shape[0]
    if entry == "plain":
        C = ops.gemm_w4a16_bf16(A, w)
    elif entry == "noalloc":
        C = ops.gemm_w4a16_bf16_noalloc(A, w, ops.empty((M, w.N), np.int16))
    else:
        C = ops.gemm_w4a16_bf16_ws(A, w, ops.w4a16_bf16_workspace(M, w) if entry == "ws" else None)
    return D.bf16_bits_to_f32(ops.host(C, np.uint16)).astype(np.float64)


def _products(x, u, z, s, G):
    s64 = np.repeat(s.astype(np.float64), G, axis=0)
    w = (u.astype(np.float64) - np.repeat(z.astype(np.float64), G, axis=0)) * s64
    a = np.abs(x).astype(np.float64)
    return x.astype(np.float64) @ w, 2.0 ** -24 * 303 * (a @ np.abs(s64)), a @ np.abs(w)


@pytest.mark.parametrize("K,N,G", [
    (128, 16, 32), (384, 33, 64), (2048, 5120, 32), (1152, 7000, 64), (1664, 13000, 32), (640, 28672, 64),
    (2176, 3000, 128), (3072, 14336, 128), (3968, 6144, 128), (2048, 8192, 256), (1536, 28672, 256), (8192, 1000, 128),
])
@pytest.mark.parametrize("Ms", [(5, 8, 9, 13, 16, 17), (24, 32, 33, 48, 49, 64)])
def test_bf16(oracle, ops, K, N, G, Ms):
    u, z, s, packed = _codes(K, N, G, K + N)
    w = ops.prepack_w4_asym(ops.dev(packed), ops.dev(s.view(np.uint16)), ops.dev(z), K, N, G)
    xb = D.to_bf16_bits(oracle, D.normal((64, K), 1.0, K))
    want, unit, _ = _products(D.bf16_bits_to_f32(xb), u, z, s, G)
    for M in Ms:
        A = ops.dev(np.ascontiguousarray(xb[:M]))
        outs = {e: _bf16_call(ops, e, A, w) for e in ("plain", "ws", "none", "noalloc")}
        for e, got in outs.items():
            _check_bf16(got, want[:M], unit[:M], K, G, (M, e))
        if _form(ops, M, N, K, G):  # no workspace is used: one result
            assert np.array_equal(outs["ws"], outs["none"]) and np.array_equal(outs["ws"], outs["noalloc"]), M


def _check_bf16(got, want, unit, K, G, what):
    assert np.isfinite(got).all(), what
    assert (np.abs(got - want) <= (2 * K + 2 * K // G + 8) * unit + 2.0 ** -8 * np.abs(want)).all(), what
    assert np.linalg.norm(got - want) <= 2.5e-3 * np.linalg.norm(want), what


# every form: 16-row blocks x column tiles per workgroup, at each number of
# scale groups per K tile (G = 32, 64, 128 and more); live rows, K tiles and
# columns ragged
FORMS = [
    (15, 1152, 4000, 1, 1), (9, 1664, 8100, 1, 2), (14, 2176, 14336, 1, 4),
    (24, 1664, 6500, 2, 2), (31, 1408, 16000, 2, 4),
    (48, 1152, 8000, 4, 2), (61, 1920, 14500, 4, 4),
]


@pytest.mark.parametrize("M,K,N,rb,ct", FORMS)
@pytest.mark.parametrize("G", [32, 64, 128, 384])
def test_every_form_bf16(oracle, ops, M, K, N, rb, ct, G):
    K = K // G * G
    assert _form(ops, M, N, K, G) == (rb, ct)
    u, z, s, packed = _codes(K, N, G, K + N)
    w = ops.prepack_w4_asym(ops.dev(packed), ops.dev(s.view(np.uint16)), ops.dev(z), K, N, G)
    xb = D.to_bf16_bits(oracle, D.normal((M, K), 1.0, K))
    want, unit, _ = _products(D.bf16_bits_to_f32(xb), u, z, s, G)
    _check_bf16(_bf16_call(ops, "ws", ops.dev(xb), w), want, unit, K, G, G)


@pytest.mark.parametrize("M,K,N,rb,ct", [(6, 1024, 4000, 1, 1), (16, 1920, 8000, 1, 2), (9, 1536, 14000, 1, 4),
                                         (17, 896, 8000, 2, 2), (32, 896, 13000, 2, 4)])
@pytest.mark.parametrize("G", [128, 384])
def test_every_form_f32(ops, M, K, N, rb, ct, G):
    K = K // G * G
    assert _form(ops, M, N, K, G, 1) == (rb, ct)
    u, _, s, packed = _codes(K, N, G, K + N)
    w = ops.prepack_w4_sym(ops.dev((packed ^ 0x88).astype(np.uint8)), ops.dev(s.astype(np.float32)), K, N, G)
    x = D.normal((M, K), 1.0, K)
    C = ops.dev(np.full((M, N), np.nan, np.float32))
    ops.run("lhq_gemm_w4a16", ops.dev(x), w.qweight, w.scales, C, M, N, K, G, 1.0, 0.0)
    got = ops.host(C).astype(np.float64)
    want, unit, mag = _products(x, u, np.full_like(u[: K // G], 8), s, G)
    bound = (4 * K + 2 * K // G + 8) * unit + 2.0 ** -17 * mag + 2.0 ** -22 * np.abs(want)
    assert (np.abs(got - want) <= bound).all()
    assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)


@pytest.mark.parametrize("K,N,G,alpha,beta", [
    (128, 16, 128, 1.0, 0.0), (1152, 300, 128, 0.5, 2.0), (1024, 14336, 128, 1.0, 0.0), (2048, 8192, 256, 1.0, -1.0),
    (8192, 1000, 128, 1.0, 0.0),
])
def test_f32(ops, K, N, G, alpha, beta):
    u, _, s, packed = _codes(K, N, G, K + N)
    s32 = s.astype(np.float32)
    w = ops.prepack_w4_sym(ops.dev((packed ^ 0x88).astype(np.uint8)), ops.dev(s32), K, N, G)  # codes as signed nibbles
    x = D.normal((32, K), 1.0, K)
    C0 = D.normal((32, N), 1.0, 5)
    prod, unit, mag = _products(x, u, np.full_like(u[: K // G], 8), s, G)
    for M in (5, 8, 9, 16, 17, 32):
        C = ops.dev(C0[:M])
        ops.run("lhq_gemm_w4a16", ops.dev(x[:M]), w.qweight, w.scales, C, M, N, K, G, alpha, beta)
        got = ops.host(C).astype(np.float64)
        want = alpha * prod[:M] + beta * C0[:M]
        bound = abs(alpha) * ((4 * K + 2 * K // G + 8) * unit[:M] + 2.0 ** -17 * mag[:M]) + 2.0 ** -22 * (
            np.abs(want) + np.abs(beta * C0[:M]))
        assert (np.abs(got - want) <= bound).all(), M
        assert np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want), M


@pytest.mark.parametrize("entry", ["plain", "ws"])
@pytest.mark.parametrize("M,K,N,G", [(17, 1152, 7000, 64), (17, 1152, 7000, 128), (17, 1152, 4000, 32)])
def test_non_finite_rows_stay_apart(oracle, ops, M, K, N, G, entry):
    assert bool(_form(ops, M, N, K, G)) == (N == 7000)
    u, z, s, packed = _codes(K, N, G, 2)
    w = ops.prepack_w4_asym(ops.dev(packed), ops.dev(s.view(np.uint16)), ops.dev(z), K, N, G)
    x = D.normal((M, K), 1.0, 3)
    x[4, 700], x[16, 1151] = np.inf, np.nan
    got = _bf16_call(ops, entry, ops.dev(D.to_bf16_bits(oracle, x)), w)
    bad = ~np.isfinite(got)
    assert bad[16].all() and bad[4].any()
    bad[[4, 16]] = False
    assert not bad.any()


@pytest.mark.parametrize("M,K,N", [(16, 8192, 8192), (8, 8192, 4096), (16, 4096, 8192)])
def test_misaligned_workspace_is_refused_as_before(ops, M, K, N):
    """Where the tiles would split K over it, a workspace that is not 16-byte
    aligned is an error, also where this kernel takes the call."""
    from longhornai_amd import capi
    G, L = 128, ops.lib()
    qw = ops.dev(np.zeros(K * ((N + 15) // 16 * 16) // 2, np.uint8))
    sc = ops.dev(np.zeros((K // G) * ((N + 15) // 16 * 16), np.float32))
    zs = ops.dev(np.zeros((K // G) * ((N + 15) // 16 * 16), np.uint8))
    A, C = ops.dev(np.zeros((M, K), np.float32)), ops.dev(np.zeros((M, N), np.float32))
    refused = 0
    for name, need, rest in [
        ("lhq_gemm_w4a16_bf16_ws", L.lhq_gemm_w4a16_bf16_workspace_bytes(M, N, K, G), ()),
        ("lhq_gemm_w4a16_ws", L.lhq_gemm_w4a16_workspace_bytes(M, N, K, G), (1.0, 0.0)),
    ]:
        if need <= 0:
            continue
        ws = ops.dev(np.zeros(need + 16, np.uint8))
        weights = (qw, sc, zs) if "bf16" in name else (qw, sc)
        with pytest.raises(capi.LhqError, match="16-byte aligned"):
            ops.run(name, A, *weights, C, M, N, K, G, *rest, ws[4:], need)
        refused += 1
    assert refused
