"""The vectorised quantizers, dequantizers and prepacks at the sizes where
their splits end: odd widths, misaligned buffers, the last partial tile, the
largest row kept in registers, the one-launch limit of the per-tensor
quantizer, exact ties.  Quantizers against the CPU oracle bit for bit (they
are defined so); the prepacked layouts against a numpy statement of the
layout in include/longhorn_hip.h, byte for byte.
"""
import numpy as np
import pytest

from tests import _data as D

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops(lib):
    from longhornai_amd import ops as _ops
    return _ops


def _same(got, want):
    got, want = np.ascontiguousarray(got), np.ascontiguousarray(want)
    assert got.shape == want.shape and got.tobytes() == want.tobytes()


def _off(ops, a, lead):
    """`a` on the device, `lead` elements past an allocation's start."""
    flat = np.concatenate([np.zeros(lead, a.dtype), a.ravel()])
    return ops.dev(flat)[lead:]


def _weights(K, N, seed):
    """Normal weights with exact ties of the quotient (scale 1 for int4
    symmetric, 127 / 127 per column), a zero column, NaN and a huge value."""
    w = D.normal((K, N), 0.02, seed)
    ties = np.arange(K, dtype=np.float32) % 15 - 7 + 0.5
    w[:, 0] = np.where(ties > 6, 7.0, ties)
    if N > 4:
        w[:, 1] = 0.0
        w[::3, 2] = np.nan
        w[1, 3] = 3e38
        w[:, 4] = np.abs(w[:, 4])
    return w


@pytest.mark.parametrize("lead", [0, 1])
@pytest.mark.parametrize("K,N,G", [(64, 63, 32), (192, 65, 64), (384, 130, 128), (512, 1, 256), (96, 5, 48)])
def test_int4_groups(oracle, ops, K, N, G, lead):
    w = _weights(K, N, K + N)
    src = _off(ops, w, lead)
    p_w, s_w = oracle.q4_quantize_groupwise(w, G)
    p, s = ops.empty((K // 2, N), np.uint8), ops.empty((K // G, N), np.float32)
    ops.run("lhq_q4_quantize_groupwise", src, p, s, K, N, G)
    _same(ops.host(p), p_w)
    _same(ops.host(s), s_w)
    p_w, s_w, z_w = oracle.q4a_quantize_groupwise(w, G)
    s, z = ops.empty((K // G, N), np.int16), ops.empty((K // G, N), np.uint8)
    ops.run("lhq_q4a_quantize_groupwise", src, p, s, z, K, N, G)
    _same(ops.host(p), p_w)
    _same(ops.host(s, np.uint16), s_w)
    _same(ops.host(z), z_w)


@pytest.mark.parametrize("K,N,G", [(30, 7, 3), (30, 9, 1), (64, 1027, 16), (34, 4, 2), (10, 6, 10), (66, 1, 2), (62, 2, 1),
                                   (516, 3, 6), (2048, 1027, 16), (2052, 1026, 9)])
@pytest.mark.parametrize("lead", [0, 3])
def test_int4_dequantize(oracle, ops, K, N, G, lead):
    g = D.rng(K * N + G)
    p = g.integers(0, 256, (K // 2, N)).astype(np.uint8)
    s = D.uniform((K // G, N), 0.01, 2.0, N)
    d = ops.empty((K * N + lead,), np.float32)[lead:]
    ops.run("lhq_q4_dequantize_groupwise", _off(ops, p, lead), _off(ops, s, lead), d, K, N, G)
    _same(ops.host(d).reshape(K, N), oracle.q4_dequantize_groupwise(p, s, K, N, G))
    s16 = s.astype(np.float16).view(np.uint16)
    z = g.integers(0, 16, (K // G, N)).astype(np.uint8)
    ops.run("lhq_q4a_dequantize_groupwise", _off(ops, p, lead), _off(ops, s16, lead), _off(ops, z, lead), d, K, N, G)
    _same(ops.host(d).reshape(K, N), oracle.q4a_dequantize_groupwise(p, s16, z, K, N, G))


# 1 << 17 elements is the last one-launch size; beyond it 4096-element shares
@pytest.mark.parametrize("n", [3, 4095, 4097, (1 << 17) - 1, 1 << 17, (1 << 17) + 1, (1 << 19) + 4099])
@pytest.mark.parametrize("kind", ["q8", "fp8"])
def test_per_tensor(oracle, ops, n, kind):
    x = D.normal((n,), 1.0, n)
    x[n // 2] = np.nan
    x[n - 1] = -7.75                              # the maximum is the last element
    q_w, s_w = getattr(oracle, f"{kind}_quantize_per_tensor")(x)
    for lead in (0, 1):
        q = ops.empty((n + lead,), np.uint8)[lead:]
        s = ops.empty((1,), np.float32)
        ops.run(f"lhq_{kind}_quantize_per_tensor", _off(ops, x, lead), q, s, n)
        _same(ops.host(q), np.asarray(q_w).view(np.uint8))
        assert ops.host(s)[0] == np.float32(s_w)


def test_per_tensor_empty(ops):
    s = ops.dev(np.full(1, 7.0, np.float32))
    ops.run("lhq_q8_quantize_per_tensor", ops.empty((1,), np.float32), ops.empty((1,), np.int8), s, 0)
    assert ops.host(s)[0] == 1.0


# one row chunk (any height below 64 rows), a chunk's edges, two column blocks, a
# last word across a block's edge, narrow matrices, two and eight rows a thread
@pytest.mark.parametrize("rows,cols", [(1, 5), (2, 1030), (63, 258), (64, 3), (129, 257), (1000, 7), (16, 255), (5, 1), (9, 2),
                                       (70, 259), (2100, 510), (1025, 1030), (1 << 18, 3), ((1 << 18) + 9, 3)])
@pytest.mark.parametrize("kind", ["q8", "fp8"])
def test_per_col(oracle, ops, rows, cols, kind):
    x = _weights(rows, cols, rows * cols) if rows > 1 else D.normal((rows, cols), 1.0, cols)
    x[rows - 1, cols - 1] = 50.0
    x[:, 0] *= 127.0 / 7.0 if kind == "q8" else 1.0
    q_w, s_w = getattr(oracle, f"{kind}_quantize_per_col")(x)
    q = ops.empty((rows * cols + 1,), np.uint8)[1:]
    s = ops.empty((cols,), np.float32)
    ops.run(f"lhq_{kind}_quantize_per_col", _off(ops, x, 1), q, s, rows, cols)
    _same(ops.host(q).reshape(rows, cols), np.asarray(q_w).view(np.uint8))
    _same(ops.host(s), s_w)


# rows kept in registers, a chunk of 16 bytes or two, four, eight a thread: up to
# 1024, 2048, 4096, 8192 in fp32, twice that in bf16; longer ones read twice
@pytest.mark.parametrize("dim", [8192, 8196, 8200, 4, 8, 1024, 1028, 2048, 2052, 2056, 4096, 4104, 16384, 16392])
def test_per_row_register_limit(oracle, ops, dim):
    x = D.normal((3, dim), 1.0, dim)
    x[1, dim - 1] = 30.0
    for kind in ("q8", "fp8"):
        q_w, s_w = getattr(oracle, f"{kind}_quantize_per_row")(x)
        q, s = ops.empty((3, dim), np.uint8), ops.empty((3,), np.float32)
        ops.run(f"lhq_{kind}_quantize_per_row", x, q, s, 3, dim)
        _same(ops.host(q), np.asarray(q_w).view(np.uint8))
        _same(ops.host(s), s_w)
    xb = D.to_bf16_bits(oracle, x)
    q_w, s_w = oracle.q8_quantize_per_row_bf16(xb)
    q = ops.empty((3, dim), np.int8)
    ops.run("lhq_q8_quantize_per_row_bf16", xb, q, s, 3, dim)
    _same(ops.host(q), q_w)
    _same(ops.host(s), s_w)


def test_sizes_near_two_to_the_31(ops):
    n = (1 << 31) - 1
    x = ops.zeros((n,), np.float32)
    x[n - 1], x[5] = 50.0, -25.0
    q, s = ops.empty((n,), np.int8), ops.empty((1,), np.float32)
    ops.run("lhq_q8_quantize_per_col", x, q, s, n, 1)
    assert ops.host(s)[0] == np.float32(50.0) / np.float32(127.0)
    assert int((q != 0).sum()) == 2 and int(q[n - 1]) == 127 and int(q[5]) == -64
    x.fill_(0.5)
    x[n - 1] = 3.0
    p, d = ops.zeros((n,), np.uint8), ops.empty((2 * n,), np.float32)
    p[n - 1], p[0] = 0x7A, 0x01
    ops.run("lhq_q4_dequantize_groupwise", p, x, d, 2, n, 2)
    assert int((d != 0).sum()) == 3
    assert float(d[n - 1]) == -18.0 and float(d[2 * n - 1]) == 21.0 and float(d[0]) == 0.5


def _w4_layout(codes, K, N):
    """[Nt][Kt][64][16 B]: lane l, dword j, element e at nibble w4_slot(e)."""
    Nt, Kt = -(-N // 16), -(-K // 128)
    u = np.zeros((Kt * 128, Nt * 16), np.uint32)
    u[:K, :N] = codes
    t = u.reshape(Kt, 4, 4, 8, Nt, 16)            # kt, j, l >> 4, e, nt, l & 15
    slot = np.array([0, 2, 4, 6, 1, 3, 5, 7], np.uint32)
    d = (t << (4 * slot)[None, None, None, :, None, None]).sum(axis=3, dtype=np.uint32)
    return d.transpose(3, 0, 2, 4, 1).astype("<u4").tobytes()  # nt, kt, l >> 4, l & 15, j


@pytest.mark.parametrize("K,N,G", [(128, 16, 32), (160, 63, 32), (256, 257, 64), (384, 1030, 128), (2, 3, 2)])
@pytest.mark.parametrize("lead", [0, 1])
def test_w4_prepack_layout(ops, K, N, G, lead):
    g = D.rng(K + 7 * N)
    u = g.integers(0, 16, (K, N)).astype(np.uint8)
    packed = (u[0::2] | (u[1::2] << 4)).astype(np.uint8)
    NG, Nt = K // G, -(-N // 16)
    z = g.integers(0, 16, (NG, N)).astype(np.uint8)
    s16 = g.integers(0, 1 << 15, (NG, N)).astype(np.uint16)
    q, s, zo = ops.w4_buffers(K, N, G, True)
    ops.run("lhq_w4_prepack_asym", _off(ops, packed, lead), ops.dev(s16), _off(ops, z, lead), K, N, G, q, s, zo)
    assert ops.host(q).tobytes() == _w4_layout(u, K, N)
    want = np.zeros((NG, Nt * 16), np.uint16)
    want[:, :N] = s16
    _same(ops.host(s, np.uint16), want.reshape(NG, Nt, 16).transpose(1, 0, 2).ravel())
    want = np.zeros((-(-NG // 8) * 8, Nt * 16), np.uint32)
    want[:NG, :N] = z
    want = (want.reshape(-1, 8, Nt, 16) << (4 * np.arange(8, dtype=np.uint32))[None, :, None, None]).sum(axis=1, dtype=np.uint32)
    _same(ops.host(zo, np.uint32), want.transpose(1, 0, 2).ravel())
    sf = D.normal((NG, N), 1.0, 3)
    q, s, _ = ops.w4_buffers(K, N, G, False)
    ops.run("lhq_w4_prepack_sym", _off(ops, packed, lead), ops.dev(sf), K, N, G, q, s)
    assert ops.host(q).tobytes() == _w4_layout(u ^ 8, K, N)


@pytest.mark.parametrize("K,N", [(128, 128), (130, 257), (1, 3), (300, 1001), (128, 5), (4, 126), (700, 2), (131, 4)])
def test_b8_prepack_layout(ops, K, N):
    b = D.rng(K + N).integers(0, 256, (K, N)).astype(np.uint8)
    bt = ops.prepack_b8(_off(ops, b, 1), K, N)
    want = np.zeros((-(-N // 256) * 256, -(-K // 128) * 128), np.uint8)
    want[:N, :K] = b.T
    _same(ops.host(bt), want.ravel())
