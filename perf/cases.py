"""The performance cases of the quantized-GEMM path: what a program that uses
this library has it do, through the public entry points, with the sizes of the
repository's own benchmark configurations and generic ones beside them.

A case is a dict of plain values; its "kind" names the call sequence:

  w4       bf16 W4A16 linear layer (asymmetric int4): decode and prefill
  w4_f32   the fp32 W4A16 interface (symmetric int4, alpha), with a workspace
  w8a8     per-token int8 quantization of the activations, then the W8A8 GEMM
  fp8      per-tensor fp8 quantization of the activations, then the fp8 GEMM
  moe      a whole MoE layer: dispatch, gate / up + SwiGLU, down, combine
  weights  a checkpoint's fp32 weight to a quantized, prepacked one (load time)
  exact    int4 weights to fp32, then the fp32 GEMM: the route for group sizes
           that the int4 kernels do not take and for non-finite activations

Inputs come from the seed alone.  Quantized weights are drawn as codes and
scales (normal weights, per-group / per-column ranges), so that the reference
values in `exact` need nothing of the library.
"""
import math

import torch

from longhornai_amd import ops

G128 = 128


def listed():
    return [
        # single-stream decode, attention output projection: the smallest call
        dict(name="decode_small", kind="w4", M=1, K=4096, N=4096, G=G128),
        # single-stream decode, the largest projection of the configurations
        dict(name="decode_large", kind="w4", M=1, K=8192, N=28672, G=G128),
        # batched decode at an odd batch, down projection (K = 86 groups)
        dict(name="decode_batch", kind="w4", M=13, K=11008, N=4096, G=G128),
        # a short prompt / a chunk of mixed prefill, ragged row count
        dict(name="prefill_short", kind="w4", M=200, K=4096, N=11008, G=G128),
        # a long prompt through the largest projection: the largest call
        dict(name="prefill_long", kind="w4", M=4096, K=8192, N=28672, G=G128),
        # the reference's own fp32 interface at a decode batch
        dict(name="f32_interface", kind="w4_f32", M=16, K=8192, N=10240, G=G128),
        # W8A8 prefill with its activation quantizer
        dict(name="w8a8_prefill", kind="w8a8", M=2048, K=4096, N=14336, out="bf16"),
        # fp8 batched decode with its activation quantizer
        dict(name="fp8_decode", kind="fp8", M=24, K=4096, N=14336),
        # one MoE layer over a prefill batch, top-2 of 8 experts
        dict(name="moe_prefill", kind="moe", T=512, H=4096, I=14336, E=8, topk=2, G=G128),
        # the same layer at decode, two sequences
        dict(name="moe_decode", kind="moe", T=2, H=4096, I=14336, E=8, topk=2, G=G128),
        # loading one projection: quantize and prepack
        dict(name="weights_int4", kind="weights", K=4096, N=14336, G=G128, scheme="int4_asym"),
        # a group size outside the int4 kernels: dequantize, fp32 GEMM
        dict(name="exact_f32", kind="exact", M=100, K=4096, N=4096, G=16),
    ]


# ---- drawn cases ------------------------------------------------------------

def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A matrix width: most are multiples of 64, some of 16, some odd."""
    n, r = _log_int(rng, lo, hi), rng.random()
    if r < 0.5:
        n = max(64, n // 64 * 64)
    elif r < 0.75:
        n = max(16, n // 16 * 16)
    else:
        n |= 1
    return n


def draw(rng):
    """One more case of the ranges the listed ones stand for, at no more than
    the cost of the largest of them."""
    kind = rng.choice(["w4"] * 5 + ["w8a8"] * 3 + ["moe"] * 3 + ["w4_f32", "w4_f32", "fp8", "fp8", "weights",
                                                                 "weights", "exact"])
    if kind == "moe":
        E, topk = rng.choice([(8, 2), (8, 2), (16, 2), (64, 6)])
        H = 128 * _log_int(rng, 8, 32)
        I = 128 * _log_int(rng, 8, min(112, 3584 * 128 * 8 // (E * H)))
        return dict(kind=kind, T=_log_int(rng, 1, 512), H=H, I=I, E=E, topk=topk, G=G128)
    if kind == "weights":
        scheme = rng.choice(["int4_asym", "int4_asym", "int4_sym", "int8", "fp8"])
        G = rng.choice([32, 64, G128, G128])
        return dict(kind=kind, K=G * (_log_int(rng, 1024, 11008) // G), N=_width(rng, 1024, 14336), G=G,
                    scheme=scheme)
    if kind == "exact":
        G = rng.choice([2, 8, 16, 16])
        return dict(kind=kind, M=_log_int(rng, 1, 512), K=G * (_log_int(rng, 256, 4096) // G),
                    N=_width(rng, 256, 4096), G=G)
    if kind in ("w8a8", "fp8"):
        case = dict(kind=kind, M=_log_int(rng, 1, 4096), K=16 * _log_int(rng, 64, 512), N=_width(rng, 1024, 14336))
        if kind == "w8a8":
            case["out"] = rng.choice(["bf16", "bf16", "fp32"])
        elif rng.random() < 0.75:
            case["K"] = max(1024, case["K"] // 128 * 128)
        return case
    G = rng.choice([32, 64, G128, G128, G128, 256])
    K = G * (_log_int(rng, 1024, 14336) // G)
    # group sizes under 128 are served at decode batches
    if kind == "w4_f32":
        return dict(kind=kind, M=_log_int(rng, 1, 512 if G >= 128 else 64), K=K, N=_width(rng, 1024, 14336), G=G)
    N, top = _width(rng, 1024, 28672), 4096 if G >= 128 else 64
    return dict(kind=kind, M=max(1, min(_log_int(rng, 1, top), 4096 * 8192 * 28672 // (K * N))), K=K, N=N, G=G)


# ---- inputs -----------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _acts(g, rows, cols):
    """Activations: unit normal, each channel with a gain of its own."""
    gain = torch.exp(0.5 * torch.randn((1, cols), generator=g, device="cuda"))
    return torch.randn((rows, cols), generator=g, device="cuda").mul_(gain)


def _bits(x):
    """bf16 as the 16-bit patterns that the library's entry points take."""
    return x.to(torch.bfloat16).view(torch.int16)


def _wide(bits):
    return bits.view(torch.bfloat16).double()


def _int4_asym(g, K, N, G):
    """Codes, fp16 scales and zero points of normal weights: (packed, scales, zeros)."""
    s = (0.008 * torch.exp(0.15 * torch.randn((K // G, N), generator=g, device="cuda"))).half()
    z = torch.randn((K // G, N), generator=g, device="cuda").mul_(0.8).add_(7.5).round_().clamp_(0, 15)
    u = torch.randn((K, N), generator=g, device="cuda").mul_(2.6)
    u = u.view(K // G, G, N).add_(z[:, None, :]).round_().clamp_(0, 15).to(torch.uint8).view(K, N)
    return u[0::2] | (u[1::2] << 4), s, z.to(torch.uint8)


def _int4_sym(g, K, N, G):
    s = 0.008 * torch.exp(0.15 * torch.randn((K // G, N), generator=g, device="cuda"))
    q = torch.randn((K, N), generator=g, device="cuda").mul_(2.6).round_().clamp_(-7, 7)
    u = q.to(torch.int8).view(torch.uint8) & 15
    return u[0::2] | (u[1::2] << 4), s


def _codes(packed):
    K, N = 2 * packed.shape[0], packed.shape[1]
    u = torch.empty((K, N), dtype=torch.uint8, device="cuda")
    u[0::2], u[1::2] = packed & 15, packed >> 4
    return u


def _dense_asym(packed, s, z, G):
    u = _codes(packed)
    K, N = u.shape
    return (u.view(K // G, G, N).double().sub_(z[:, None, :].double()).mul_(s[:, None, :].double())).view(K, N)


def _dense_sym(packed, s, G):
    u = _codes(packed).to(torch.int8)
    K, N = u.shape
    q = torch.where(u > 7, u - 16, u)
    return (q.view(K // G, G, N).double().mul_(s[:, None, :].double())).view(K, N)


def _int8_cols(g, K, N):
    q = torch.randn((K, N), generator=g, device="cuda").mul_(31.0).round_().clamp_(-127, 127).to(torch.int8)
    return q, 6e-4 * torch.exp(0.2 * torch.randn((N,), generator=g, device="cuda"))


def _routing(g, case):
    """Experts of uneven popularity, and the gates of a softmax over the chosen ones."""
    T, E, topk = case["T"], case["E"], case["topk"]
    scores = torch.randn((T, E), generator=g, device="cuda") + 0.5 * torch.randn((1, E), generator=g, device="cuda")
    top = torch.topk(scores, topk, dim=1)
    return top.indices.to(torch.int32).contiguous(), torch.softmax(top.values, dim=1).contiguous()


def _moe_weights(case, seed):
    """Per expert: gate [H, I], up [H, I], down [I, H] as int4 codes."""
    H, I, G = case["H"], case["I"], case["G"]
    for e in range(case["E"]):
        g = _gen(seed * 1000003 + 17 + e)
        yield _int4_asym(g, H, I, G), _int4_asym(g, H, I, G), _int4_asym(g, I, H, G)


def _fp8_weights(g, K, N):
    w = torch.randn((K, N), generator=g, device="cuda").mul_(0.02 * 448.0 / 0.11).clamp_(-448, 448)
    return w.to(torch.float8_e4m3fn).view(torch.uint8), torch.full((1,), 0.11 / 448.0, device="cuda")


def _buf(shape, dtype):
    return torch.empty(shape, dtype=dtype, device="cuda")


# ---- a case's state ---------------------------------------------------------

def prepare(case, seed):
    kind, g = case["kind"], _gen(seed)
    if kind == "moe":
        return _prepare_moe(case, seed, g)
    K, N = case["K"], case["N"]
    if kind == "weights":
        w = torch.randn((K, N), generator=g, device="cuda").mul_(0.02)
        st = dict(case=case, w=w)
        if case["scheme"].startswith("int4"):
            asym = case["scheme"] == "int4_asym"
            st["packed"] = _buf((K // 2, N), torch.uint8)
            st["scales"] = _buf((K // case["G"], N), torch.int16 if asym else torch.float32)
            st["zeros"] = _buf((K // case["G"], N), torch.uint8) if asym else None
        else:
            st["codes"] = _buf((K, N), torch.uint8)
            st["scales"] = _buf((N,) if case["scheme"] == "int8" else (1,), torch.float32)
        return st
    M = case["M"]
    if kind == "w4":
        w = ops.prepack_w4_asym(*_bits16(_int4_asym(g, K, N, case["G"])), K, N, case["G"])
        return dict(case=case, a=_bits(_acts(g, M, K)), w=w, ws=ops.w4a16_bf16_workspace(M, w),
                    c=_buf((M, N), torch.int16))
    if kind == "w4_f32":
        w = ops.prepack_w4_sym(*_int4_sym(g, K, N, case["G"]), K, N, case["G"])
        nbytes = ops.lib().lhq_gemm_w4a16_workspace_bytes(M, N, K, case["G"])
        return dict(case=case, a=_acts(g, M, K), w=w, ws=_buf((nbytes,), torch.uint8) if nbytes > 0 else None,
                    nbytes=nbytes, c=_buf((M, N), torch.float32))
    if kind == "w8a8":
        q, s = _int8_cols(g, K, N)
        x, bf16 = _acts(g, M, K), case["out"] == "bf16"
        return dict(case=case, bt=ops.prepack_b8(q, K, N), bs=s, x=_bits(x) if bf16 else x,
                    aq=_buf((M, K), torch.int8), as_=_buf((M,), torch.float32),
                    c=_buf((M, N), torch.int16 if bf16 else torch.float32))
    if kind == "fp8":
        b8, bs = _fp8_weights(g, K, N)
        return dict(case=case, bt=ops.prepack_b8(b8, K, N), bs=bs, x=_acts(g, M, K), a8=_buf((M, K), torch.uint8),
                    as_=_buf((1,), torch.float32), c=_buf((M, N), torch.float32))
    packed, s = _int4_sym(g, K, N, case["G"])
    return dict(case=case, packed=packed, scales=s, a=_acts(g, M, K), w=_buf((K, N), torch.float32),
                c=_buf((M, N), torch.float32))


def _bits16(w):
    return w[0], w[1].view(torch.int16), w[2]


def _prepare_moe(case, seed, g):
    T, H, I, E, topk, G = (case[k] for k in ("T", "H", "I", "E", "topk", "G"))
    ids, gates = _routing(g, case)
    x = _bits(_acts(g, T, H))
    gate_up, down = [], []
    for wg, wu, wd in _moe_weights(case, seed):
        gate_up.append(ops.interleave_gate_up(ops.prepack_w4_asym(*_bits16(wg), H, I, G),
                                              ops.prepack_w4_asym(*_bits16(wu), H, I, G)))
        down.append(ops.prepack_w4_asym(*_bits16(wd), I, H, G))
    S = T * topk
    L = ops.lib()
    nbytes = max(L.lhq_gemm_w4a16_bf16_grouped_swiglu_workspace_bytes(E, S, I, H, G),
                 L.lhq_gemm_w4a16_bf16_grouped_workspace_bytes(E, S, H, I, G))
    return dict(case=case, x=x, ids=ids, gates=gates, gate_up=gate_up, down=down,
                tables=ops.pointer_tables(gate_up) + ops.pointer_tables(down),
                offsets=_buf((E + 1,), torch.int32), token=_buf((S,), torch.int32), slot=_buf((S,), torch.int32),
                pos=_buf((S,), torch.int32), xs=_buf((S, H), torch.int16), act=_buf((S, I), torch.int16),
                y=_buf((S, H), torch.int16), out=_buf((T, H), torch.int16),
                ws=_buf((nbytes,), torch.uint8) if nbytes > 0 else None, nbytes=nbytes)


# ---- one pass ---------------------------------------------------------------

def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "w4":
        return ops.gemm_w4a16_bf16_ws(st["a"], st["w"], st["ws"], st["c"]).view(torch.bfloat16)
    if kind == "w4_f32":
        w = st["w"]
        ops.run("lhq_gemm_w4a16_ws", st["a"], w.qweight, w.scales, st["c"], case["M"], w.N, w.K, w.G, 0.5, 0.0,
                st["ws"], st["nbytes"])
        return st["c"]
    if kind == "moe":
        return _run_moe(st, case)
    if kind == "weights":
        return _run_weights(st, case)
    M, N, K = case["M"], case["N"], case["K"]
    if kind == "w8a8":
        if case["out"] == "bf16":
            ops.run("lhq_q8_quantize_per_row_bf16", st["x"], st["aq"], st["as_"], M, K)
            c = ops.gemm_w8a8_bf16(st["aq"], st["bt"], st["as_"], st["bs"], M, N, K, st["c"]).view(torch.bfloat16)
        else:
            ops.run("lhq_q8_quantize_per_row", st["x"], st["aq"], st["as_"], M, K)
            c = ops.gemm_w8a8(st["aq"], st["bt"], st["as_"], st["bs"], M, N, K, st["c"], alpha=0.5)
        return st["aq"], st["as_"], c
    if kind == "fp8":
        ops.run("lhq_fp8_quantize_per_tensor", st["x"], st["a8"], st["as_"], M * K)
        ops.run("lhq_gemm_fp8_e4m3", st["a8"], st["bt"], st["as_"], st["bs"], st["c"], M, N, K, 1.0, 0.0)
        return st["a8"], st["as_"], st["c"]
    ops.run("lhq_q4_dequantize_groupwise", st["packed"], st["scales"], st["w"], K, N, case["G"])
    ops.run("lhq_gemm_f32", st["a"], st["w"], st["c"], M, N, K, 1.0, 0.0)
    return st["w"], st["c"]


def _run_moe(st, case):
    T, H, I, E, topk, G = (case[k] for k in ("T", "H", "I", "E", "topk", "G"))
    ops.run("lhq_moe_dispatch_bf16", st["x"], st["ids"], st["offsets"], st["token"], st["slot"], st["pos"],
            st["xs"], T, H, E, topk)
    ops.run("lhq_moe_expert_mlp_w4a16_bf16_ws", st["xs"], st["offsets"], *st["tables"], st["act"], st["y"], E,
            T * topk, H, I, G, st["ws"], st["nbytes"])
    ops.run("lhq_moe_combine_bf16", st["y"], st["pos"], st["gates"], st["out"], T, H, topk)
    return (st["offsets"], st["token"], st["slot"], st["pos"], st["act"].view(torch.bfloat16),
            st["y"].view(torch.bfloat16), st["out"].view(torch.bfloat16))


def _run_weights(st, case):
    K, N, G, scheme = case["K"], case["N"], case["G"], case["scheme"]
    if scheme == "int4_asym":
        ops.run("lhq_q4a_quantize_groupwise", st["w"], st["packed"], st["scales"], st["zeros"], K, N, G)
        p = ops.prepack_w4_asym(st["packed"], st["scales"], st["zeros"], K, N, G)
        return st["packed"], st["scales"].view(torch.float16), st["zeros"], p.qweight, p.scales, p.zeros
    if scheme == "int4_sym":
        ops.run("lhq_q4_quantize_groupwise", st["w"], st["packed"], st["scales"], K, N, G)
        p = ops.prepack_w4_sym(st["packed"], st["scales"], K, N, G)
        return st["packed"], st["scales"], p.qweight, p.scales
    if scheme == "int8":
        ops.run("lhq_q8_quantize_per_col", st["w"], st["codes"], st["scales"], K, N)
    else:
        ops.run("lhq_fp8_quantize_per_tensor", st["w"], st["codes"], st["scales"], K * N)
    return st["codes"], st["scales"], ops.prepack_b8(st["codes"], K, N)


# ---- what a pass cannot do without -----------------------------------------

def _int4_bytes(K, N, G, asym):
    return K * N / 2 + (K / G) * N * (2.5 if asym else 4)


def work(case):
    kind = case["kind"]
    if kind == "moe":
        T, H, I, E, topk, G = (case[k] for k in ("T", "H", "I", "E", "topk", "G"))
        S = T * topk
        used = E * (1.0 - (1.0 - topk / E) ** T)  # experts with a token, expected
        weights = used * (2 * _int4_bytes(H, I, G, True) + _int4_bytes(I, H, G, True))
        rows = 2 * (T * H + S * H + S * I + S * H + T * H)
        return dict(bytes=weights + rows + 4 * (5 * S + E + 1), flops=6.0 * S * H * I + 2.0 * S * H)
    K, N = case["K"], case["N"]
    if kind == "weights":
        if case["scheme"].startswith("int4"):
            return dict(bytes=4 * K * N + 2 * _int4_bytes(K, N, case["G"], case["scheme"] == "int4_asym"),
                        flops=2.0 * K * N)
        return dict(bytes=6 * K * N + 4 * (N if case["scheme"] == "int8" else 1), flops=2.0 * K * N)
    M = case["M"]
    flops = 2.0 * M * K * N
    if kind == "w4":
        return dict(bytes=_int4_bytes(K, N, case["G"], True) + 2 * M * (K + N), flops=flops)
    if kind == "w4_f32":
        return dict(bytes=_int4_bytes(K, N, case["G"], False) + 4 * M * (K + N), flops=flops)
    if kind == "w8a8":
        act, out = (2, 2) if case["out"] == "bf16" else (4, 4)
        return dict(bytes=K * N + M * K * (act + 1) + 4 * (M + N) + out * M * N, flops=flops)
    if kind == "fp8":
        return dict(bytes=K * N + 5 * M * K + 4 * M * N + 8, flops=flops)
    return dict(bytes=_int4_bytes(K, N, case["G"], False) + 4 * K * N + 4 * M * (K + N), flops=flops + K * N)


def tolerance(case):
    """Quantizers, W8A8 and the fp32 dequantizer are defined bit for bit.  The
    others: about four times what the path differs by from `exact`."""
    return {
        "w4": {"rel": 7e-3},       # one rounding to bf16 (1.7e-3)
        "w4_f32": {"rel": 2.5e-5}, # bf16 hi + lo activations, fp32 sums (6e-6)
        "fp8": {"rel": 8e-5},      # the sums inside the fp8 matrix instructions (2e-5)
        "moe": {"rel": 1.2e-2},    # bf16 between the projections and at the end (2.9e-3)
        "exact": {"rel": 4.5e-6},  # fp32 sums (1.1e-6)
    }.get(case["kind"], "exact")


# ---- the same in 64 bits, in plain torch ------------------------------------

# Which code a value gets is defined by fp32 steps: scale = max / 127 (or 448),
# then x * (1 / scale) per row and per tensor, x / scale per column.

def _scale(m, top):
    """max / top in one fp32 rounding (torch multiplies by a constant's reciprocal)."""
    return torch.where(m > 0, (m.double() / top).float(), torch.ones_like(m))


def _per_row(x):
    s = _scale(x.abs().amax(dim=1), 127.0)
    return (x * (1.0 / s)[:, None]).round().clamp(-127, 127).double(), s


def _per_tensor(x):
    s = _scale(x.abs().max(), 448.0).reshape(1)
    return _e4m3(x * (1.0 / s)), s


def _e4m3(x):
    """Round to e4m3 (saturating at 448, nothing below 2^-9); doubles come back."""
    x = torch.where(x.abs() < 2.0 ** -9, 0.0, x).double().clamp(-448.0, 448.0)
    e = torch.floor(torch.log2(x.abs().clamp_min(2.0 ** -60))).clamp_min(-6.0)
    step = torch.exp2(e - 3.0)
    return (x / step).round() * step


def _e4m3_bits(v):
    return v.to(torch.float32).to(torch.float8_e4m3fn).view(torch.uint8)


def exact(case, seed):
    kind = case["kind"]
    if kind == "moe":
        return _exact_moe(case, seed)
    if kind == "weights":
        return _exact_weights(case, seed)
    g, M, K, N = _gen(seed), case["M"], case["K"], case["N"]
    if kind == "w4":
        w = _dense_asym(*_int4_asym(g, K, N, case["G"]), case["G"])
        return _wide(_bits(_acts(g, M, K))) @ w
    if kind == "w4_f32":
        w = _dense_sym(*_int4_sym(g, K, N, case["G"]), case["G"])
        return 0.5 * (_acts(g, M, K).double() @ w)
    if kind == "w8a8":
        b, bs = _int8_cols(g, K, N)
        x, bf16 = _acts(g, M, K), case["out"] == "bf16"
        q, s = _per_row(_wide(_bits(x)).float() if bf16 else x)
        c = (q @ b.double()) * s.double()[:, None] * bs.double()[None, :]
        return q.to(torch.int8), s, c if bf16 else 0.5 * c
    if kind == "fp8":
        b8, bs = _fp8_weights(g, K, N)
        a, s = _per_tensor(_acts(g, M, K))
        return _e4m3_bits(a), s, (a @ b8.view(torch.float8_e4m3fn).double()) * (s.double() * bs.double())
    w = _dense_sym(*_int4_sym(g, K, N, case["G"]), case["G"])
    return w, _acts(g, M, K).double() @ w


def _exact_moe(case, seed):
    T, H, E, topk, G = (case[k] for k in ("T", "H", "E", "topk", "G"))
    g = _gen(seed)
    ids, gates = _routing(g, case)
    x = _wide(_bits(_acts(g, T, H)))
    flat = ids.flatten().long()
    order = torch.argsort(flat, stable=True)
    offsets = torch.zeros(E + 1, dtype=torch.int64, device="cuda")
    offsets[1:] = torch.cumsum(torch.bincount(flat, minlength=E), 0)
    pos = torch.empty_like(order)
    pos[order] = torch.arange(order.numel(), device="cuda")
    act = torch.empty((T * topk, case["I"]), dtype=torch.float64, device="cuda")
    y = torch.empty((T * topk, H), dtype=torch.float64, device="cuda")
    bounds = offsets.tolist()
    for e, (wg, wu, wd) in enumerate(_moe_weights(case, seed)):
        lo, hi = bounds[e], bounds[e + 1]
        if hi > lo:
            rows = x[order[lo:hi] // topk]
            act[lo:hi] = torch.nn.functional.silu(rows @ _dense_asym(*wg, G)) * (rows @ _dense_asym(*wu, G))
            y[lo:hi] = act[lo:hi] @ _dense_asym(*wd, G)
    out = (y[pos].view(T, topk, H) * gates.double()[:, :, None]).sum(dim=1)
    whole = [v.to(torch.int32) for v in (offsets, order // topk, order % topk, pos)]
    return (*whole, act, y, out)


def _exact_weights(case, seed):
    """Scales and codes; the prepacked layouts hold the same values again."""
    K, N, G, scheme = case["K"], case["N"], case["G"], case["scheme"]
    w = torch.randn((K, N), generator=_gen(seed), device="cuda").mul_(0.02)
    if scheme == "int8":
        s = _scale(w.abs().amax(dim=0), 127.0)
        return (w / s).round().clamp(-127, 127).to(torch.int8).view(torch.uint8), s, None
    if scheme == "fp8":
        v, s = _per_tensor(w)
        return _e4m3_bits(v), s, None
    grouped = w.view(K // G, G, N)
    if scheme == "int4_sym":
        s = _scale(grouped.abs().amax(dim=1), 7.0)
        u = (grouped / s[:, None, :]).round().clamp(-7, 7).to(torch.int8).view(torch.uint8).view(K, N) & 15
        return u[0::2] | (u[1::2] << 4), s, None, None
    lo, hi = grouped.amin(dim=1).clamp_max(0.0), grouped.amax(dim=1).clamp_min(0.0)
    s = _scale(hi - lo, 15.0).half().float().clamp_min(2.0 ** -14)
    z = (-lo / s).round().clamp(0, 15)
    u = ((grouped / s[:, None, :]).round() + z[:, None, :]).clamp(0, 15).to(torch.uint8).view(K, N)
    return u[0::2] | (u[1::2] << 4), s, z.to(torch.uint8), None, None, None
