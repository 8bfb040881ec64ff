"""The 64 x 256 bf16 tile of the W4A16 prefill on 32x32x16 MFMAs: shapes with
ragged last rows and columns around its row count, G = 128 and 256, batches,
and scales that vary as far as fp16 goes, vanish or are all zero, under
ordinary and very large activations.

Tolerance, against float64 on the same codes: inside a group a partial sum of a
column never exceeds 303 sum_k |x| (terms x (144 + u - z) and -144 x), the
group's sum is then multiplied by its scale (exactly 0 for a zero scale, so
such a group adds nothing, rounding errors included) and added, and each of the
K + 4 K/G additions and products rounds once (2^-24), so
|error| <= 2^-24 (K + 4 K/G) 303 sum_k s |x|, plus half an ulp of bf16 (2^-8
|want|).  Relative Frobenius: bf16 rounding alone is at most 2^-9, so 2.5e-3.
"""
import numpy as np
import pytest

from tests import _data as D

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops(lib):
    from longhornai_amd import ops as _ops
    return _ops


def _case(M, N, K, G, seed, scales=None):
    g = D.rng(seed)
    u = g.integers(0, 16, (K, N)).astype(np.uint8)
    z = g.integers(0, 16, (K // G, N)).astype(np.uint8)
    s = (0.01 * np.exp(0.3 * g.standard_normal((K // G, N)))).astype(np.float16) if scales is None else scales
    x = D.normal((M, K), 1.0, seed + 1)
    return u, z, s, x


def _prepack(ops, u, z, s, K, N, G):
    packed = (u[0::2] | (u[1::2] << 4)).astype(np.uint8)
    return ops.prepack_w4_asym(ops.dev(packed), ops.dev(s.view(np.uint16)), ops.dev(z), K, N, G)


def _check(got, x, u, z, s, G):
    K = u.shape[0]
    s64 = np.repeat(s.astype(np.float64), G, axis=0)
    w = (u.astype(np.float64) - np.repeat(z.astype(np.float64), G, axis=0)) * s64
    want = x.astype(np.float64) @ w
    bound = 2.0 ** -24 * (K + 4 * K // G) * 303 * (np.abs(x).astype(np.float64) @ np.abs(s64)) + 2.0 ** -8 * np.abs(want)
    assert np.isfinite(got).all()
    assert (np.abs(got - want) <= bound).all()
    return np.linalg.norm(got - want) / max(np.linalg.norm(want), 1e-300)


# 8 row tiles at two widths, 7 with one row over, 8 x 17, one row tile, one
# row past a tile
@pytest.mark.parametrize("M,N,K,G", [(450, 28700, 256, 128), (512, 28672, 512, 256), (385, 28672, 128, 128),
                                     (449, 4100, 384, 128), (64, 20000, 256, 128), (65, 40000, 512, 256)])
def test_shapes(oracle, ops, M, N, K, G):
    u, z, s, x = _case(M, N, K, G, M + K)
    xb = D.to_bf16_bits(oracle, x)
    w = _prepack(ops, u, z, s, K, N, G)
    got = D.bf16_bits_to_f32(ops.host(ops.gemm_w4a16_bf16(ops.dev(xb), w), np.uint16)).astype(np.float64)
    assert _check(got, D.bf16_bits_to_f32(xb), u, z, s, G) <= 2.5e-3


@pytest.mark.parametrize("M,N,batch", [(256, 4100, 14), (130, 300, 3)])
def test_batched(oracle, ops, M, N, batch):
    K, G = 256, 128
    cs = [_case(M, N, K, G, 7 * b) for b in range(batch)]
    xb = [D.to_bf16_bits(oracle, c[3]) for c in cs]
    ws = [_prepack(ops, *c[:3], K, N, G) for c in cs]
    import torch
    q, s, z = (torch.cat([getattr(w, f) for w in ws]) for f in ("qweight", "scales", "zeros"))
    C = ops.empty((batch, M, N), np.int16)
    ops.run("lhq_gemm_w4a16_bf16_batched", np.stack(xb), q, s, z, C, batch, M, N, K, G)
    got = D.bf16_bits_to_f32(ops.host(C, np.uint16)).astype(np.float64)
    for b in (0, batch - 1):
        assert _check(got[b], D.bf16_bits_to_f32(xb[b]), *cs[b][:3], G) <= 2.5e-3


def _hard_scales(NG, N, seed):
    """Column classes: zeros between and before ordinary scales, all zero,
    alternating 6e-8 and 6e4, rising and falling over the whole fp16 range,
    negative, equal."""
    g = D.rng(seed)
    s = (0.01 * np.exp(0.3 * g.standard_normal((NG, N)))).astype(np.float16)
    c = np.arange(N) % 8
    s[:, c == 0] = np.where(g.random((NG, (c == 0).sum())) < 0.5, 0, s[:, c == 0])
    s[: NG // 2, c == 1] = 0
    s[:, c == 2] = 0
    s[:, c == 3] = np.where(np.arange(NG) % 2, 6e-8, 6e4).astype(np.float16)[:, None]
    s[:, c == 4] = (6e-8 * (1e12 ** (np.arange(NG) / max(NG - 1, 1)))).clip(6e-8, 6.5e4).astype(np.float16)[:, None]
    s[:, c == 5] = s[:, c == 4][::-1][:, : (c == 5).sum()]
    s[:, c == 6] *= np.float16(-1)
    s[:, c == 7] = np.float16(0.0123)
    return s


# two row tiles, eight, and a split-K launch
@pytest.mark.parametrize("M,N,K", [(80, 16400, 1024), (450, 28672, 1024), (64, 4096, 8192)])
def test_scale_range(oracle, ops, M, N, K):
    G = 128
    u, z, s, x = _case(M, N, K, G, K, _hard_scales(K // G, N, 3))
    xb = D.to_bf16_bits(oracle, x)
    w = _prepack(ops, u, z, s, K, N, G)
    C = ops.gemm_w4a16_bf16_ws(ops.dev(xb), w, ops.w4a16_bf16_workspace(M, w))
    got = D.bf16_bits_to_f32(ops.host(C, np.uint16)).astype(np.float64)
    xf = D.bf16_bits_to_f32(xb)
    _check(got, xf, u, z, s, G)
    assert (got[:, np.arange(N) % 8 == 2] == 0).all()


# the same launches: groups of zero scale hold activations up to 1e8 times the
# others'
@pytest.mark.parametrize("M,N,K", [(80, 16400, 1024), (450, 28672, 1024), (64, 4096, 8192)])
def test_zero_scaled_groups_add_nothing(oracle, ops, M, N, K):
    G = 128
    u, z, s, x = _case(M, N, K, G, K + 1)
    g = D.rng(K)
    dead = np.arange(K // G) % 3 == 1
    s[dead] = 0
    x *= np.where(dead, g.choice([1e6, 1e7, 1e8], K // G), 1.0).astype(np.float32).repeat(G)
    xb = D.to_bf16_bits(oracle, x)
    w = _prepack(ops, u, z, s, K, N, G)
    C = ops.gemm_w4a16_bf16_ws(ops.dev(xb), w, ops.w4a16_bf16_workspace(M, w))
    got = D.bf16_bits_to_f32(ops.host(C, np.uint16)).astype(np.float64)
    assert _check(got, D.bf16_bits_to_f32(xb), u, z, s, G) <= 2.5e-3


def test_non_finite_scales_and_rows(oracle, ops):
    M, N, K, G = 450, 28672, 512, 128
    u, z, s, x = _case(M, N, K, G, 9)
    u[:, :64] = (z[:, :64].repeat(G, axis=0) + 1) % 16
    s[1, 3], s[2, 7], s[3, 100] = np.inf, np.nan, np.inf
    x[5, 17], x[200, 300] = np.inf, np.nan
    w = _prepack(ops, u, z, s, K, N, G)
    got = D.bf16_bits_to_f32(ops.host(ops.gemm_w4a16_bf16(ops.dev(D.to_bf16_bits(oracle, x)), w), np.uint16))
    bad = ~np.isfinite(got)
    assert np.isnan(got[[5, 200]]).all() and bad[:, [3, 7, 100]].all()
    bad[[5, 200]] = False
    bad[:, [3, 7, 100]] = False
    assert not bad.any()
