// prepack.hip -- one-time re-tiling of quantized weights into the layouts the
// gfx950 GEMM kernels stream.
//
// The reference keeps int4 weights as [K/2, N] bytes (quant.hpp:52-59) and
// int8 weights as [K, N] (gemm_quant.hpp:37), and reads them with a stride of
// N bytes per k step (gemm_quant.cpp:42, quant.hpp:71).  On the GPU that
// stride would make every wave touch K/2 separate rows for one column; these
// kernels rewrite the weights once so each wave reads contiguous 1 KiB runs
// that are already in MFMA operand order.
#include "common.hpp"

namespace lhq {
namespace {

// Eight codes of four adjacent columns are four packed rows (k / 2) of four
// bytes: r[i] holds rows i of a 32-bit word per column quad.  Rewritten to
// the operand order of the layout (w4_slot: byte i of a column's dword is
// element i in the low nibble and element 4 + i in the high one), still one
// byte per column; a 4x4 byte transpose then gives each column its dword.
__device__ __forceinline__ void w4_quad(const uint32_t (&r)[4], uint32_t (&out)[4]) {
    constexpr uint32_t L = 0x0F0F0F0Fu, H = 0xF0F0F0F0u;
    const uint32_t b0 = (r[0] & L) | ((r[2] & L) << 4);  // elements 0, 4
    const uint32_t b1 = ((r[0] >> 4) & L) | (r[2] & H);  // elements 1, 5
    const uint32_t b2 = (r[1] & L) | ((r[3] & L) << 4);  // elements 2, 6
    const uint32_t b3 = ((r[1] >> 4) & L) | (r[3] & H);  // elements 3, 7
    const uint32_t x0 = __builtin_amdgcn_perm(b1, b0, 0x05010400u), x1 = __builtin_amdgcn_perm(b1, b0, 0x07030602u);
    const uint32_t y0 = __builtin_amdgcn_perm(b3, b2, 0x05010400u), y1 = __builtin_amdgcn_perm(b3, b2, 0x07030602u);
    out[0] = __builtin_amdgcn_perm(y0, x0, 0x05040100u);
    out[1] = __builtin_amdgcn_perm(y0, x0, 0x07060302u);
    out[2] = __builtin_amdgcn_perm(y1, x1, 0x05040100u);
    out[3] = __builtin_amdgcn_perm(y1, x1, 0x07060302u);
}

// One launch for the whole prepack.  Workgroups [0, qblocks) re-tile the
// codes: wave v of a workgroup owns K tile kt and the 64 columns from
// 64 * v of a 256-column block.  Lane (c4 = l & 15, kq = l >> 4) reads, as
// 32-bit words, columns 4 c4 .. + 3 of the 16 packed rows that hold its k
// values of the four 32-deep blocks, and writes the 16-byte chunks of lanes
// 16 kq + 4 (c4 & 3) .. + 3 of the column tile: 64 contiguous bytes, 1 KiB
// per four-column-tile store over the wave.  The remaining workgroups copy
// the scales and pack the zero points, one element per thread.
// Bound by memory: K=4096, N=14336 moves 2 x 30 MB.  (A thread per output
// chunk reading sixteen single bytes, and three launches, took 55.5 us on
// the GPU; this 18.5.)  Rows past K and columns past N become zero codes.  Any N and
// alignment: a row's words may be misaligned, and a quad that crosses the
// last column reads its bytes one by one.
template <bool ASYM, typename S>
__global__ __launch_bounds__(256) void w4_prepack_kernel(const uint8_t* __restrict__ packed,
                                                         uint8_t* __restrict__ qweight,
                                                         const S* __restrict__ scales, S* __restrict__ scales_out,
                                                         const uint8_t* __restrict__ zeros,
                                                         uint32_t* __restrict__ zeros_out, int K, int N, int Nt,
                                                         int Kt, int NG, int64_t qblocks, int64_t sblocks) {
    const int64_t blk = static_cast<int64_t>(blockIdx.y) * gridDim.x + blockIdx.x;
    if (blk < qblocks) {
        const int kt = static_cast<int>(blk % Kt);
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        const int c4 = lane & 15, kq = lane >> 4;
        const int n0 = static_cast<int>(blk / Kt) * 256 + wave * 64 + 4 * c4;
        const int nt = n0 / kW4TileN;
        if (nt >= Nt) return;
        const int rows = K / 2;
        uint32_t d[4][4];  // [32-deep block][column]
        auto read = [&](auto full) {
            const int cnt = full.value ? 4 : max(N - n0, 0);
            // symmetric: two's-complement q in [-8,7] -> q + 8 (quant.hpp:73-74), live columns only
            const uint32_t flip = ASYM ? 0u : 0x88888888u & (full.value ? 0xFFFFFFFFu : (1u << (8 * (cnt & 3))) - 1u);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                uint32_t r[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int row = kt * (kW4TileK / 2) + 16 * j + 4 * kq + i;
                    r[i] = load_u8x4<full.value>(packed + static_cast<int64_t>(min(row, rows - 1)) * N + n0, cnt) ^ flip;
                    r[i] = row < rows ? r[i] : 0u;
                }
                w4_quad(r, d[j]);
            }
        };
        if (n0 <= N - 4) read(Full{});
        else read(Part{});
        u32x4_t* o = reinterpret_cast<u32x4_t*>(qweight + (static_cast<int64_t>(nt) * Kt + kt) * kW4TileBytes) +
                     16 * kq + 4 * (c4 & 3);
#pragma unroll
        for (int c = 0; c < 4; ++c) o[c] = u32x4_t{d[0][c], d[1][c], d[2][c], d[3][c]};
        return;
    }
    if (blk < qblocks + sblocks) {
        const int64_t t = (blk - qblocks) * 256 + threadIdx.x;
        if (t >= static_cast<int64_t>(Nt) * NG * 16) return;
        const int64_t r = t >> 4;
        const int g = static_cast<int>(r % NG);
        const int n = static_cast<int>(r / NG) * kW4TileN + static_cast<int>(t & 15);
        scales_out[t] = (n < N) ? scales[static_cast<int64_t>(g) * N + n] : S(0);
        return;
    }
    if constexpr (ASYM) {
        const int NG8 = (NG + 7) / 8;
        const int64_t t = (blk - qblocks - sblocks) * 256 + threadIdx.x;
        if (t >= static_cast<int64_t>(Nt) * NG8 * 16) return;
        const int64_t r = t >> 4;
        const int g8 = static_cast<int>(r % NG8);
        const int n = static_cast<int>(r / NG8) * kW4TileN + static_cast<int>(t & 15);
        uint32_t v = 0;
        if (n < N) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int g = g8 * 8 + i;
                if (g < NG) v |= (static_cast<uint32_t>(zeros[static_cast<int64_t>(g) * N + n]) & 0xfu) << (4 * i);
            }
        }
        zeros_out[t] = v;
    }
}

template <bool ASYM, typename S>
int launch_w4_prepack(const uint8_t* packed, const S* scales, const uint8_t* zeros, int K, int N, int G,
                      uint8_t* qweight, S* scales_out, uint32_t* zeros_out, hipStream_t s, const char* who) {
    const int Nt = ceil_div(N, kW4TileN), Kt = ceil_div(K, kW4TileK), NG = K / G;
    const int64_t qb = static_cast<int64_t>(ceil_div(Nt, 16)) * Kt;
    const int64_t sb = ceil_div64(static_cast<int64_t>(Nt) * NG * 16, 256);
    const int64_t zb = ASYM ? ceil_div64(static_cast<int64_t>(Nt) * ceil_div(NG, 8) * 16, 256) : 0;
    // a second grid dimension past 2^30 threads; the blocks past the last one end
    // in the last section's own bounds
    const int64_t total = qb + sb + zb, gx = total < (1 << 22) ? total : 1 << 22;
    w4_prepack_kernel<ASYM, S><<<dim3(static_cast<unsigned>(gx), static_cast<unsigned>(ceil_div64(total, gx))), 256, 0, s>>>(
        packed, qweight, scales, scales_out, zeros, zeros_out, K, N, Nt, Kt, NG, qb, sb);
    return check_launch(who);
}

// Bt[n][k] = B[k][n] for n < N, k < K, zero elsewhere.  A workgroup
// transposes 128 k x 128 n through LDS: a thread reads four rows of four
// adjacent columns as 32-bit words (128 contiguous bytes per row and eight
// lanes' rows at a time), transposes the 4x4 bytes in registers and puts
// four k of one column in LDS as one word; the write-out then stores 16
// bytes of k per lane, 128 contiguous bytes per column.  The odd row stride
// keeps the transposed words of a wave within two to a bank.
// Bound by memory: K=4096, N=14336 moves 2 x 58.7 MB in 19 us a call (6.2
// TB/s; a 64x64 tile moved byte by byte took 48).
__global__ __launch_bounds__(256) void b8_prepack_kernel(const uint8_t* __restrict__ B,
                                                        uint8_t* __restrict__ Bt, int K, int N,
                                                        int Kp) {
    __shared__ uint32_t tile[128][33];  // [column][word of four k], one word of padding
    const int k0 = blockIdx.x * 128, n0 = blockIdx.y * 128;
    const int c4 = threadIdx.x & 31;
    const int n = n0 + 4 * c4;
    const int cnt = max(N - n, 0);
    // words past the last column are read from column N - 4 on (K=1024, N=411
    // 2.5 us; 5.0 byte by byte in their own branch)
    const int from = N >= 4 ? min(n, N - 4) : n, shift = 8 * min(n - from, 3);
    auto put = [&](auto full) {
        uint32_t r[4][4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int k = k0 + 4 * (static_cast<int>(threadIdx.x >> 5) + 8 * u) + i;
                const uint32_t v = load_u8x4<full.value>(B + static_cast<int64_t>(min(k, K - 1)) * N + from, cnt);
                r[u][i] = k < K && cnt > 0 ? v >> shift : 0u;
            }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int kw = (threadIdx.x >> 5) + 8 * u;  // word of k: rows 4 kw .. + 3
            const uint32_t x0 = __builtin_amdgcn_perm(r[u][1], r[u][0], 0x05010400u);
            const uint32_t x1 = __builtin_amdgcn_perm(r[u][1], r[u][0], 0x07030602u);
            const uint32_t y0 = __builtin_amdgcn_perm(r[u][3], r[u][2], 0x05010400u);
            const uint32_t y1 = __builtin_amdgcn_perm(r[u][3], r[u][2], 0x07030602u);
            tile[4 * c4 + 0][kw] = __builtin_amdgcn_perm(y0, x0, 0x05040100u);
            tile[4 * c4 + 1][kw] = __builtin_amdgcn_perm(y0, x0, 0x07060302u);
            tile[4 * c4 + 2][kw] = __builtin_amdgcn_perm(y1, x1, 0x05040100u);
            tile[4 * c4 + 3][kw] = __builtin_amdgcn_perm(y1, x1, 0x07060302u);
        }
    };
    if (N >= 4) put(Full{});
    else put(Part{});
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int col = (threadIdx.x >> 3) + 32 * u, w = 4 * (threadIdx.x & 7);
        const u32x4_t v = {tile[col][w], tile[col][w + 1], tile[col][w + 2], tile[col][w + 3]};
        __builtin_memcpy(Bt + static_cast<int64_t>(n0 + col) * Kp + k0 + 4 * w, &v, 16);
    }
}

// Interleave two prepacked W4 tensors by column tile: output block 2i is
// block i of `a`, block 2i + 1 is block i of `b` (a block is everything one
// column tile owns: blk16 16-byte units).  One 16-byte copy per thread.
__global__ void w4_interleave_kernel(const u32x4_t* __restrict__ a, const u32x4_t* __restrict__ b,
                                     u32x4_t* __restrict__ out, int64_t blk16, int64_t total16) {
    const int64_t d = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (d >= total16) return;
    const int64_t blk = d / blk16, off = d - blk * blk16;
    const u32x4_t* src = (blk & 1) ? b : a;
    out[d] = src[(blk >> 1) * blk16 + off];
}

int launch_interleave(const void* a, const void* b, void* out, int64_t blk_bytes, int tiles, hipStream_t s) {
    const int64_t blk16 = blk_bytes / 16, total16 = 2 * blk16 * tiles;
    if (total16 == 0) return LHQ_OK;
    w4_interleave_kernel<<<static_cast<unsigned>(ceil_div64(total16, 256)), 256, 0, s>>>(
        static_cast<const u32x4_t*>(a), static_cast<const u32x4_t*>(b), static_cast<u32x4_t*>(out), blk16, total16);
    return check_launch("w4_interleave_gate_up");
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

}  // namespace lhq

using namespace lhq;

extern "C" {

int lhq_w4_prepack_sym(const uint8_t* packed, const float* scales, int K, int N, int G,
                       uint8_t* qweight, float* scales_out, void* stream) {
    LHQ_REQUIRE(packed && scales && qweight && scales_out, "w4_prepack_sym: null pointer");
    LHQ_REQUIRE(w4_dims_ok(K, N, G), "w4_prepack_sym: need K,N,G > 0, K even, G | K (K=%d N=%d G=%d)", K, N, G);
    return launch_w4_prepack<false>(packed, scales, nullptr, K, N, G, qweight, scales_out, nullptr, as_stream(stream),
                                    "w4_prepack_sym");
}

int lhq_w4_prepack_asym(const uint8_t* packed, const uint16_t* scales_f16, const uint8_t* zeros,
                        int K, int N, int G, uint8_t* qweight, uint16_t* scales_out,
                        uint32_t* zeros_out, void* stream) {
    LHQ_REQUIRE(packed && scales_f16 && zeros && qweight && scales_out && zeros_out,
                "w4_prepack_asym: null pointer");
    LHQ_REQUIRE(w4_dims_ok(K, N, G), "w4_prepack_asym: need K,N,G > 0, K even, G | K (K=%d N=%d G=%d)", K, N, G);
    return launch_w4_prepack<true>(packed, scales_f16, zeros, K, N, G, qweight, scales_out, zeros_out,
                                   as_stream(stream), "w4_prepack_asym");
}

int lhq_w4_interleave_gate_up(const uint8_t* gate_qweight, const uint16_t* gate_scales,
                              const uint32_t* gate_zeros, const uint8_t* up_qweight,
                              const uint16_t* up_scales, const uint32_t* up_zeros, int K, int I, int G,
                              uint8_t* qweight, uint16_t* scales_out, uint32_t* zeros_out, void* stream) {
    LHQ_REQUIRE(gate_qweight && gate_scales && gate_zeros && up_qweight && up_scales && up_zeros && qweight &&
                    scales_out && zeros_out,
                "w4_interleave_gate_up: null pointer");
    LHQ_REQUIRE(w4_dims_ok(K, I, G), "w4_interleave_gate_up: need K,I,G > 0, K even, G | K (K=%d I=%d G=%d)", K, I,
                G);
    const void* all[9] = {gate_qweight, gate_scales, gate_zeros, up_qweight, up_scales, up_zeros,
                          qweight,      scales_out,  zeros_out};
    for (const void* ptr : all) LHQ_REQUIRE(aligned16(ptr), "w4_interleave_gate_up: pointers must be 16-byte aligned");
    const int Nt = ceil_div(I, kW4TileN), Kt = ceil_div(K, kW4TileK), NG = K / G, NG8 = ceil_div(NG, 8);
    hipStream_t s = as_stream(stream);
    if (int st = launch_interleave(gate_qweight, up_qweight, qweight, static_cast<int64_t>(Kt) * kW4TileBytes, Nt, s))
        return st;
    if (int st = launch_interleave(gate_scales, up_scales, scales_out, static_cast<int64_t>(NG) * kW4TileN * 2, Nt, s))
        return st;
    return launch_interleave(gate_zeros, up_zeros, zeros_out, static_cast<int64_t>(NG8) * kW4TileN * 4, Nt, s);
}

int64_t lhq_b8_prepacked_bytes(int K, int N) {
    if (K <= 0 || N <= 0) return 0;
    return static_cast<int64_t>(ceil_div(N, 256)) * 256 * (static_cast<int64_t>(ceil_div(K, 128)) * 128);
}

int lhq_b8_prepack(const uint8_t* B, int K, int N, uint8_t* Bt, void* stream) {
    LHQ_REQUIRE(B && Bt, "b8_prepack: null pointer");
    LHQ_REQUIRE(K > 0 && N > 0, "b8_prepack: need K, N > 0 (K=%d N=%d)", K, N);
    const int Kp = ceil_div(K, 128) * 128, Np = ceil_div(N, 256) * 256;
    dim3 grid(Kp / 128, Np / 128);
    b8_prepack_kernel<<<grid, 256, 0, as_stream(stream)>>>(B, Bt, K, N, Kp);
    return check_launch("b8_prepack");
}

}  // extern "C"
