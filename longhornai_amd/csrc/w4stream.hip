// w4stream.hip -- W4A16 for a few rows: 5..64 in bf16 (the workspace and the
// no-allocation entry points; lhq_gemm_w4a16_bf16 and the batched and grouped
// ones keep the kernels beside it), 5..32 of the fp32 interface, where
// w4_stream_rb finds it the fastest.
//
// The weights' read bounds these calls (K=8192, N=28672 at G=32: 132 MB, 20 us
// at 6.5 TB/s), and below about 20 MB of weights the launch.  The kernels
// beside this one lose to it in two ways: the 16-row kernel reads its
// activations from L2 beside the weights, 64 bytes of 16 rows at a time and
// four times the weights' bytes; the tiles split over K write and read back
// fp32 partial sums and launch twice.  Here a workgroup of eight waves, CT
// 16-column tiles x KP = 8 / CT parts of K, stages its rows once, a phase of
// KCT K tiles at a time into one of two LDS buffers (bf16 by DMA, whole 1 KiB
// runs of a row; fp32 through registers, split into bf16 hi and lo planes),
// and each wave keeps a window of eight weight tiles with their scales and
// zero points in flight from its first tile to its last: a tile's registers
// are reloaded as soon as it is consumed.  What grows with the rows is that
// staging, which every workgroup repeats from L2.
//
// Measured before and now, us (bf16 unless said):
//   G=32,  K=8192, N=28672:  M=8 41.3 / 34.9, M=24 70.7 / 54.0, M=64 134 / 84
//   G=64,  K=4096, N=14336:  M=16 15.3 / 11.0, M=32 20.3 / 14.4, M=64 30.7 / 20.8
//   G=128, K=4096, N=14336:  M=8 14.4 / 10.2, M=16 12.7 / 10.9
//   G=128, K=2048, N=5120:   M=16 9 / 6.6, M=64 13 / 9
//   G=128, K=14336, N=4096:  M=16 17.4 / 13.4
//   fp32,  K=2048, N=12288:  M=16 14.1 / 9.4, M=24 13.5 / 13.0
//   fp32,  K=1024, N=8192:   M=24 12.0 / 7.3
//
// Per tile and 16-row block the chain t = sum_k x (144 + u - z) + sum_k x (-144)
// (MFMAs on exact bf16 integers, the zero point folded into the codes) is
// sum_k x (u - z), and acc += s t: the arithmetic of the other kernels, per
// group of at most 128 k.  The K parts meet in LDS in K order: results are
// deterministic.
#include <algorithm>

#include "w4common.hpp"

namespace lhq {
namespace {

constexpr int kWindow = 8;  // weight tiles in flight per wave
constexpr int kWaves = 8;

// K tiles per phase: 64 KiB of LDS per buffer at 16 RB rows
constexpr int phase_tiles(bool f32, int RB) { return (f32 ? 8 : 16) / RB; }

template <bool F32, int RB, int CT, int BPS>
__global__ __launch_bounds__(64 * kWaves, 2) void w4_stream_kernel(W4Args p) {
    constexpr int KP = kWaves / CT, KCT = phase_tiles(F32, RB), SP = KCT / KP;  // SP: a wave's tiles of a phase
    constexpr int SEGS = 4 / BPS;                    // scale groups per K tile
    static_assert(SP >= 1 && kWindow % SP == 0, "a window holds whole phases");
    constexpr int LPT = 1 + SEGS + (F32 ? 0 : 1);    // loads per tile
    constexpr int PITCH = KCT * kW4TileK * (F32 ? 4 : 2);  // LDS bytes per row: per K tile 256 of bf16, or of hi then lo
    constexpr int TB = kW4TileK * (F32 ? 4 : 2);
    extern __shared__ __attribute__((aligned(1024))) uint8_t lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ct = wave % CT, kp = wave / CT;
    const int r16 = lane & 15, kg = lane >> 4;
    const int nt_wave = static_cast<int>(blockIdx.x) * CT + ct, nt = min(nt_wave, p.Nt - 1);

    const int rows = p.M;  // <= 16 RB

    auto extent = [](int64_t bytes) {
        return static_cast<int>(static_cast<uint32_t>(bytes < int64_t{0xFFFFFFFF} ? bytes : int64_t{0xFFFFFFFF}));
    };
    constexpr int ES = F32 ? 4 : 2;  // scale bytes
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(p.qw) + static_cast<int64_t>(nt) * p.Kt * kW4TileBytes, 0,
        extent(static_cast<int64_t>(p.Kt) * kW4TileBytes), kBufWord3);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        static_cast<uint8_t*>(const_cast<void*>(p.scales)) + static_cast<int64_t>(nt) * p.NG * 16 * ES, 0,
        extent(static_cast<int64_t>(p.NG) * 16 * ES), kBufWord3);
    const __amdgpu_buffer_rsrc_t rz = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint32_t*>(p.zeros) + (F32 ? 0 : static_cast<int64_t>(nt) * p.NG8 * 16), 0,
        extent(F32 ? 0 : static_cast<int64_t>(p.NG8) * 64), kBufWord3);

    // --- the weight window: the wave's tiles i = 0, 1, ... are tile i % SP of
    // its part of phase i / SP (past the end: the last one, never used)
    u32x4_t b[kWindow];
    uint32_t sw[kWindow][SEGS], zw[kWindow];
    const int phases = (p.Kt + KCT - 1) / KCT;
    int pf_phase = 0, pf_j = 0;
    auto fetch = [&](int u) {
        const int kt = min(pf_phase * KCT + kp * SP + pf_j, p.Kt - 1);
        if (++pf_j == SP) {
            pf_j = 0;
            ++pf_phase;
        }
        const int g0 = BPS < 4 ? kt * SEGS : group_of<4>(kt, 0, p.gmul);
        b[u] = __builtin_amdgcn_raw_buffer_load_b128(rw, lane * 16, kt * kW4TileBytes, 0);
#pragma unroll
        for (int s = 0; s < SEGS; ++s) {
            if constexpr (F32) sw[u][s] = __builtin_amdgcn_raw_buffer_load_b32(rs, r16 * 4, (g0 + s) * 64, 0);
            else sw[u][s] = __builtin_amdgcn_raw_buffer_load_b16(rs, r16 * 2, (g0 + s) * 32, 0);
        }
        // the tile's groups share a word: SEGS divides 8
        if constexpr (!F32) zw[u] = __builtin_amdgcn_raw_buffer_load_b32(rz, r16 * 4, (g0 >> 3) * 64, 0);
    };

    // --- the activations of a phase
    const int buf_bytes = rows * PITCH;
    const int kend = p.Kt * kW4TileK;  // K % 128 == 0
    const uint16_t* const A16 = static_cast<const uint16_t*>(p.A);
    const float* const A32 = static_cast<const float*>(p.A);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint16_t*>(A16), 0, extent(static_cast<int64_t>(rows) * p.K * 2), kBufWord3);
    auto stage = [&](int phase) {  // bf16
        const int k0 = phase * KCT * kW4TileK;
        uint8_t* const buf = lds + (phase & 1) * buf_bytes;
        for (int r = wave; r < rows; r += kWaves)
#pragma unroll
            for (int c0 = 0; c0 < PITCH / 16; c0 += 64) {
                const int k = min(k0 + 8 * ((c0 + lane) ^ (r & 15)), kend - 8);  // (past K: not used)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    ra, (LHQ_LDS_AS void*)(buf + r * PITCH + c0 * 16), 16,
                    (static_cast<uint32_t>(r) * static_cast<uint32_t>(p.K) + static_cast<uint32_t>(k)) * 2, 0, 0, 0);
            }
    };
    constexpr int CHT = F32 ? 16 * RB * KCT * 16 / (64 * kWaves) : 1;  // 8-float chunks per thread and phase
    f32x4_t fa[CHT][2];
    auto load_f32 = [&](int phase) {
        const int k0 = phase * KCT * kW4TileK;
#pragma unroll
        for (int i = 0; i < CHT; ++i) {
            const int idx = i * 64 * kWaves + static_cast<int>(threadIdx.x);
            const int r = min(idx / (KCT * 16), rows - 1), k = min(k0 + 8 * (idx % (KCT * 16)), kend - 8);
            const float* q = A32 + static_cast<int64_t>(r) * p.K + k;
            fa[i][0] = *reinterpret_cast<const f32x4_any_t*>(q);
            fa[i][1] = *reinterpret_cast<const f32x4_any_t*>(q + 4);
        }
    };
    auto split_f32 = [&](int phase) {
        uint8_t* const buf = lds + (phase & 1) * buf_bytes;
#pragma unroll
        for (int i = 0; i < CHT; ++i) {
            const int idx = i * 64 * kWaves + static_cast<int>(threadIdx.x);
            const int r = idx / (KCT * 16), c = idx % (KCT * 16);
            u32x4_t hi, lo;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float v0 = fa[i][e >> 1][2 * (e & 1)], v1 = fa[i][e >> 1][2 * (e & 1) + 1];
                const uint16_t h0 = f32_to_bf16(v0), h1 = f32_to_bf16(v1);
                hi[e] = static_cast<uint32_t>(h0) | (static_cast<uint32_t>(h1) << 16);
                lo[e] = pack_bf16x2(v0 - bf16_to_f32(h0), v1 - bf16_to_f32(h1));
            }
            if (r < rows) {
                uint8_t* const o = buf + r * PITCH + (c >> 4) * TB + ((c & 15) ^ (r & 15)) * 16;
                *reinterpret_cast<u32x4_t*>(o) = hi;
                *reinterpret_cast<u32x4_t*>(o + 256) = lo;
            }
        }
    };
    // the phase's activations are in LDS and every wave is done with the
    // buffer of the phase before.  bf16: the DMAs issued at the start of the
    // phase before have landed once at most the weight loads issued since
    // (YOUNGER of them) are in flight.
    auto barrier = [&]() {
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto landed = [&](auto younger) {
        constexpr int Y = decltype(younger)::value;
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0F70 | (Y & 15) | ((Y >> 4) << 14));
        barrier();
    };

    f32x4_t acc[RB];
#pragma unroll
    for (int i = 0; i < RB; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const u32x4_t m144 = {kM144Bf16x2, kM144Bf16x2, kM144Bf16x2, kM144Bf16x2};
    // operand rows past the staged ones read the last staged row (their
    // outputs are not stored)
    uint32_t arow[RB];
#pragma unroll
    for (int i = 0; i < RB; ++i) {
        const int r = min(16 * i + r16, rows - 1);
        arow[i] = r * PITCH + ((kg ^ (r & 15)) * 16);
    }
    auto compute = [&](int u, int phase, int j) {
        const int kt = phase * KCT + kp * SP + j;
        const uint32_t base = (phase & 1) * buf_bytes + (kp * SP + j) * TB;
        const int g0 = BPS < 4 ? kt * SEGS : group_of<4>(kt, 0, p.gmul);
#pragma unroll
        for (int s = 0; s < SEGS; ++s) {
            const float scale = F32 ? __uint_as_float(sw[u][s]) : f16_to_f32(static_cast<uint16_t>(sw[u][s]));
            const uint32_t zb =
                F32 ? 0x08080808u : __builtin_amdgcn_perm(0u, 16u - ((zw[u] >> (4 * ((g0 + s) & 7))) & 15u), 0u);
            f32x4_t t[RB];
#pragma unroll
            for (int i = 0; i < RB; ++i) t[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < BPS; ++q) {
                const int blk = s * BPS + q;
                const u32x4_t bq = w4_operand_z(b[u][blk], zb);
#pragma unroll
                for (int i = 0; i < RB; ++i) {
                    // chunk 4 blk + kg of the row's K tile (slot ^ r)
                    const uint32_t at = base + (arow[i] ^ (64 * blk));
                    const u32x4_t a = *reinterpret_cast<const u32x4_t*>(lds + at);
                    t[i] = mfma_bf16_16x16x32(a, m144, t[i]);
                    t[i] = mfma_bf16_16x16x32(a, bq, t[i]);
                    if constexpr (F32) {
                        const u32x4_t al = *reinterpret_cast<const u32x4_t*>(lds + at + 256);
                        t[i] = mfma_bf16_16x16x32(al, m144, t[i]);
                        t[i] = mfma_bf16_16x16x32(al, bq, t[i]);
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[i][e] = __builtin_fmaf(scale, t[i][e], acc[i][e]);
        }
    };

    const int total = phases * SP, groups = (total + kWindow - 1) / kWindow;
    if constexpr (F32) load_f32(0);
    else stage(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < kWindow; ++u) fetch(u);
    __builtin_amdgcn_sched_barrier(0);
    auto open = [&](int phase, auto younger) {  // the start of a phase, in every wave alike
        if constexpr (F32) {
            split_f32(phase);
            barrier();
            if (phase + 1 < phases) load_f32(phase + 1);
        } else {
            landed(younger);
            if (phase + 1 < phases) stage(phase + 1);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    open(0, std::integral_constant<int, kWindow * LPT>{});
    // one copy of the window's code, looped: it is fetched once per CU, and a
    // short call would otherwise wait for instructions rather than weights
#pragma unroll 1
    for (int gi = 0; gi < groups; ++gi) {
#pragma unroll
        for (int u = 0; u < kWindow; ++u) {
            const int i = gi * kWindow + u, phase = i / SP;  // (SP is a power of two)
            if (i < total) {
                if (u % SP == 0 && i > 0) open(phase, std::integral_constant<int, SP * LPT>{});
                if (phase * KCT + kp * SP + u % SP < p.Kt) compute(u, phase, u % SP);
            }
            fetch(u);
        }
    }

    // --- the K parts, in K order: red[kp][ct][i][lane]
    f32x4_t* const red = reinterpret_cast<f32x4_t*>(lds);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < RB; ++i) red[((kp * CT + ct) * RB + i) * 64 + lane] = acc[i];
    __syncthreads();
    // wave w stores row block w / CT.. of its column tile: CT x RB blocks over
    // eight waves
    for (int x = wave; x < CT * RB; x += kWaves) {
        const int xc = x % CT, i = x / CT;
        f32x4_t v = red[(xc * RB + i) * 64 + lane];
#pragma unroll
        for (int w = 1; w < KP; ++w) {
            const f32x4_t o = red[((w * CT + xc) * RB + i) * 64 + lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += o[e];
        }
        const int cn = (static_cast<int>(blockIdx.x) * CT + xc) * kW4TileN + r16;
        if (cn >= p.N) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int row = 16 * i + 4 * kg + e;
            if (row < p.M) w4_store<F32>(p, static_cast<int64_t>(row) * p.N + cn, v[e]);
        }
    }
}

template <bool F32, int RB, int CT, int BPS>
int launch(const W4Args& a, hipStream_t s, const char* who) {
    constexpr int pitch = phase_tiles(F32, RB) * kW4TileK * (F32 ? 4 : 2);
    constexpr size_t red = static_cast<size_t>(kWaves) * RB * 1024;
    static const hipError_t attr =
        hipFuncSetAttribute(reinterpret_cast<const void*>(&w4_stream_kernel<F32, RB, CT, BPS>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (attr != hipSuccess)
        return set_error(LHQ_ERR_HIP, "%s: dynamic LDS attribute: %s", who, hipGetErrorString(attr));
    const int rows = a.M, bufs = a.Kt > phase_tiles(F32, RB) ? 2 : 1;
    const size_t bytes = std::max(red, static_cast<size_t>(bufs) * rows * pitch);
    w4_stream_kernel<F32, RB, CT, BPS><<<ceil_div(a.Nt, CT), 64 * kWaves, bytes, s>>>(a);
    return check_launch(who);
}

template <bool F32, int RB, int BPS>
int launch_ct(const W4Args& a, int ct, hipStream_t s, const char* who) {
    constexpr int most = phase_tiles(F32, RB);  // KP = 8 / CT <= KCT
    if constexpr (8 <= most)
        if (ct == 1) return launch<F32, RB, 1, BPS>(a, s, who);
    if constexpr (4 <= most)
        if (ct == 2) return launch<F32, RB, 2, BPS>(a, s, who);
    return launch<F32, RB, 4, BPS>(a, s, who);
}

template <bool F32, int BPS>
int launch_rb(const W4Args& a, int rb, int ct, hipStream_t s, const char* who) {
    if (rb == 1) return launch_ct<F32, 1, BPS>(a, ct, s, who);
    if constexpr (!F32)
        if (rb == 4) return launch_ct<F32, 4, BPS>(a, ct, s, who);
    return launch_ct<F32, 2, BPS>(a, ct, s, who);
}

}  // namespace

namespace {

// Column tiles per workgroup: the shortest rounds of the CUs, a round being
// its tiles and the staging of the rows (about two tiles' time).  One tile
// each at N=28672 (7 rounds, M=16, K=8192) takes 57 us, four (2 rounds) 36.
int column_tiles(const W4Args& a, bool f32, int rb, int cus) {
    const int most = phase_tiles(f32, rb);
    auto cost = [&](int c) { return ceil_div(ceil_div(a.Nt, c), cus) * (c + 2); };
    int ct = 4;
    for (int c = 2; c >= 1 && 8 / c <= most; c /= 2)
        if (cost(c) < cost(ct)) ct = c;
    return ct;
}

// Where this kernel is the fastest, from 36,839 shapes timed with it and with
// the kernels beside it (those / this, us): with this rule the mean over all
// of them is 0.93 / 0.88 / 0.84 of theirs (G = 128, 64, 32; fp32 0.84), and about
// one in a thousand is 2 to 5% slower.  Every workgroup stages the rows, about two column tiles' time,
// growing with M K; a round of the CUs that is barely begun is lost; and the
// 16-row kernel, which gives a workgroup one column tile and two waves' worth
// of K each, is at its best where the tiles just fill a round of two (or, up
// to 14 rows, one) per CU.
bool stream_wins(const W4Args& a, bool f32, int ct) {
    const int M = a.M, K = a.K, G = a.G, cus = std::max(w4_device_cus(), 1);
    const int rounds = ceil_div(ceil_div(a.Nt, ct), cus);
    const int u = static_cast<int>(ceil_div64(int64_t{a.Nt} * 64, cus));  // 64ths of a column tile per CU
    const bool one = rounds == 1, full = 4 * int64_t{a.Nt} >= int64_t{3} * rounds * ct * cus;
    const bool fine = G < kW4TileK;          // several scale groups per K tile
    const bool brief = K > 512 && K < 1024;  // five to seven K tiles over eight waves
    if (f32) {  // twice the bytes to stage, and coarse groups only
        // M=17, N=12288: K=2048 13.8 / 11.7; N=1024, M=32, K=768 5.5 / 5.9
        if (M > 16) return (one && K <= 1024 && (K == 1024 || u > 32)) || (u <= 192 && K > 1024 && K <= 2048);
        // M=16: K=2048, N=14336 14.4 / 9.2; K=4096, N=8192 13.1 / 10.9; K=14336, N=512 38.9 / 21.2
        if ((M == 5 || M == 9) && K > 1024 && K < 1280) return false;
        if (M > 8) return (one && K <= 2048) || (u <= 128 && K <= 4096) || u <= 32;
        // M=5, N=4096: K=768 4.0 / 4.1, K=2304 5.4 / 5.9, K=4096 7.3 / 7.4, K=5632 16.3 / 9.4
        if (ct == 1 && ((K > 1024 && K <= 2304) || (M == 5 ? K < 5120 : M <= 7 && K > 3072 && K < (M == 6 ? 4480 : 4096))))
            return false;
        if (ct == 4 && M <= 7 && K < 1024) return false;
        return (one && K <= 4096) || (u <= 64 && K <= 8192) || u <= 32;
    }
    if (M <= 8) {
        // four tiles each: M=8, N=14336: K=4096 14.5 / 10.6, but K=5120 12.2 / 13.3
        if (ct != 4 || !full) return false;
        if (!one)
            return !fine     ? K >= 8192  // N=28672: M=8 31.6 / 31.1
                   : G == 64 ? K > 5632 || (u > 384 && K > 2048 && K <= 4096)
                             : K > 2048;
        if (!fine) return K > 2560 && u > 200 && K <= (M <= 6 ? 5120 : 4096) && (M > 6 || u <= 240);
        if (M <= 6) return K > (G == 64 ? 2048 : 3072) && (u > 200 || K > 5120);
        return K > 2048 && (u > 200 || K > 3072);
    }
    if (M <= 16) {
        if (!one) return full && K > 1024 && K <= 2048;  // N=28672, M=16: K=2048 16.5 / 11.2, K=4096 20.6 / 21.0
        if (brief && M <= 10 && ct != 2 && u <= 192) return false;
        if (ct == 2) {
            // M=13, K=7168: N=7168 14.7 / 11.6, but with the round full N=8192 11.1 / 12.2
            if (u > 124 && K > 2048) return false;
            if (!fine) return !(M <= 10 && K > 4096 && K <= 4864 && u > 100);
            return M > (G == 64 ? 10 : 12) || (K >= 1024 && !(G == 64 && K > 4096 && K <= 4608));
        }
        if (ct == 4) {
            // M=16, N=12288: K=2560 9.4 / 8.7 (M=13 slower), K=4096 12.9 / 10.7, K=14336 24.6 / 28.0
            if (!fine) return K <= 2048 || (full && (M <= 10 ? K <= 4096 : (K > 3072 && K <= 4096) || (M <= 14 && K <= 2304)));
            return G == 64 ? M > 10 || !brief : M > 12 ? !brief : K >= 1536;
        }
        // one tile each: M=9, N=4096: K=2048 4.8 / 4.7, K=5632 6.1 / 6.9; M=16: any
        if (!fine) {
            if (M <= 10) return (K <= 4096 && !(K > 1536 && K < 2048)) || u <= 16;
            if (M <= 14 && K > 4096 && K < 4608) return false;
            return M > 14 || u <= (M <= 12 ? 40 : 16) || !(K > (M <= 12 ? 4096 : 3584) && K <= 5632);
        }
        if (G == 64) {
            if (M <= 10) return K > 2304 && K <= 4608;
            return M > 14 || !(K > (M <= 12 ? 4096 : 3072) && K <= 5632);
        }
        if (M <= 12) return (K > 2304 && K <= 3584) || K > 5632;
        return !brief && !(K > 3584 && K <= 4608) && (M > 14 || !((K > 1024 && K < 1536) || (K > 1792 && K <= 2304)));
    }
    // under 1.5 tiles per CU the 16-row kernel wins to 47 rows (K=N=4096, M=32
    // 7.4 / 8.4; M=33, K=1024, N=2048 3.6 / 5.5), this one from 48 (K=2048, N=3072
    // 12.3 / 7.9)
    if (u < 96) return M >= 48 && one && K <= 2048 && !fine;
    if (M <= 32) {
        if (fine) return (one || full) && (K >= 768 || u > 124);  // G=32, M=24, K=4096, N=28672 40.6 / 30.4
        // M=17, N=7168: K=512 4.1 / 4.4, K=1536 6.4 / 6.1, K=2304 7.0 / 7.4
        if (u <= 124) return K >= 1024 && K <= 4096 && !(M <= 24 && K > 1792 && K <= 2304);
        // M=32: K=2048, N=16384 14.2 / 10.1; N=8192: K=4096 14.4 / 11.1, K=8192 16.8 / 18.3
        return (one && K <= 2048) || (rounds == 2 && K >= 512 && K <= 1024) || (u <= 128 && K <= 4096);
    }
    // a second pair of tiles for a few CUs only: M=48, G=64, K=8192: N=10240 34.2 / 41.0, N=11008 49.5 / 41.4
    const bool gap = u > 128 && u <= 170;
    if (fine) return (one || (full && !(G == 64 && K >= 8192))) && !(G == 64 && M < 64 && K >= 2048 && gap);
    // M=64, N=14336: K=2048 19.6 / 12.9, K=4096 20.8 / 22.0, K=8192 31.8 / 39.1
    return (one && K <= 2048 && !(M < 48 && K > 1536 && gap)) || (u <= 128 && K <= 4096);
}

}  // namespace

int w4_stream_rb(const W4Args& a, bool f32) {
    const int M = a.M, K = a.K, rb = M <= 16 ? 1 : M <= 32 ? 2 : 4;
    // whole K tiles; 16-byte loads of the rows; row offsets within 32 bits
    if (M < 5 || M > (f32 ? 32 : 64) || K % kW4TileK != 0 || (f32 && a.G < kW4TileK) ||
        (reinterpret_cast<uintptr_t>(a.A) & 15) != 0 || static_cast<int64_t>(M) * K * (f32 ? 4 : 2) >= (int64_t{1} << 31))
        return 0;
    const int env = tuning_knob("LHQ_W4S", -1);  // 0: never; 1: always
    if (env == 0 || env == 1) return env ? rb : 0;
    return stream_wins(a, f32, column_tiles(a, f32, rb, std::max(w4_device_cus(), 1))) ? rb : 0;
}

int launch_w4_stream(const W4Args& a, bool f32, int rb, hipStream_t s, const char* who) {
    const int ct = column_tiles(a, f32, rb, std::max(w4_device_cus(), 1));
    if (f32) return launch_rb<true, 4>(a, rb, ct, s, who);
    if (a.G == 32) return launch_rb<false, 1>(a, rb, ct, s, who);
    if (a.G == 64) return launch_rb<false, 2>(a, rb, ct, s, who);
    return launch_rb<false, 4>(a, rb, ct, s, who);
}

}  // namespace lhq

extern "C" int lhq_selftest_w4_stream(int M, int N, int K, int G, int f32) {
    using namespace lhq;
    if (M <= 0 || N <= 0 || K <= 0 || G <= 0) return 0;
    W4Args a{};
    a.M = M;
    a.N = N;
    a.K = K;
    a.G = G;
    a.Nt = ceil_div(N, kW4TileN);
    const int rb = w4_stream_rb(a, f32 != 0);
    return rb ? 16 * rb + column_tiles(a, f32 != 0, rb, std::max(w4_device_cus(), 1)) : 0;
}
