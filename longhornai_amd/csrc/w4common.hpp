// w4common.hpp -- what the W4A16 kernels share: their arguments, scale groups,
// the ragged group table, operand and output elements (w4a16.hip,
// w4stream.hip).
#pragma once

#include "common.hpp"

namespace lhq {

constexpr uint32_t kM144Bf16x2 = 0xC310C310u;  // bf16 pair (-144.0, -144.0), exact

struct W4Args {
    const void* A;
    const uint8_t* qw;
    const void* scales;
    const uint32_t* zeros;
    void* C;
    int M, N, K, G, Nt, Kt, NG, NG8;
    // group of tile kt when G > 128: __umulhi(kt, gmul), gmul = ceil(2^32 / (G/128))
    // (exact for kt, G/128 < 2^16); 0 when G <= 128
    uint32_t gmul;
    float alpha, beta;
    // per-matrix strides for uniform batches (grid.z): elements of A / C,
    // bytes of qweight, elements of scales / zeros
    int64_t a_bs, c_bs, qw_bs, s_bs, z_bs;
    // ragged groups (device-resident table): rows [offsets[e], offsets[e+1])
    // use weights qws[e], scs[e], zss[e]; num_groups == 0 means not grouped
    const int32_t* offsets;
    const uint8_t* const* qws;
    const void* const* scs;
    const uint32_t* const* zss;
    int num_groups, row_capacity;
    int group_rb;  // rows per row block of a grouped decode launch
    // split-K tile launches (grid.z = split): split s covers K tiles
    // [s * kps, (s + 1) * kps) and writes fp32 partial sums ws[s][M][N]
    float* ws;
    int kps;
    // persistent grouped launches: the workspace's 64 KiB partial-sum slots
    // (at ws) and the launch's worker count
    int64_t pk_slots;
    int pk_workers;
};

// Scale group of segment s of K tile kt; a segment is BPS 32-wide k blocks
// (min(G,128) k values), so G <= 128 needs no division at all.
template <int BPS>
__device__ __forceinline__ int group_of(int kt, int s, uint32_t gmul) {
    if constexpr (BPS < 4) return kt * (4 / BPS) + s;
    else return gmul ? static_cast<int>(__umulhi(static_cast<uint32_t>(kt), gmul)) : kt;
}
// The same with G > 128 known at compile time (GBIG) or known false.
template <int BPS, bool GBIG>
__device__ __forceinline__ int group_of_c(int kt, int s, uint32_t gmul) {
    if constexpr (BPS < 4) return kt * (4 / BPS) + s;
    else if constexpr (GBIG) return static_cast<int>(__umulhi(static_cast<uint32_t>(kt), gmul));
    else return kt;
}

// The group of a segment as read from the scale / zero arrays: with G < 128
// and K % 128 != 0 the last K tile has segments past K (their activations
// are zero), and their scale and zero point are read from the last group so
// every load stays inside the arrays.
template <int BPS, bool GBIG>
__device__ __forceinline__ int seg_group(int kt, int s, const W4Args& p) {
    const int g = group_of_c<BPS, GBIG>(kt, s, p.gmul);
    if constexpr (BPS < 4) return min(g, p.NG - 1);
    else return g;
}

// Map blockIdx.y of a grouped launch to (group, first row, row end): groups
// take ceil(rows/RB) row blocks each, in order.  Offsets are clamped to
// [0, row_capacity] so a malformed table can never index outside A or C.
// The wave resolves 64 groups per step: lane i takes group e0 + i, a prefix
// sum over the lanes gives each group's first block, and a ballot finds the
// group holding block y (4 steps for 256 experts, where a serial walk of the
// table by every workgroup cost milliseconds per layer).  The results are
// the same in every lane and wave (y is uniform): the return is uniform per
// workgroup.  rb: rows per block (a compile-time constant through
// resolve_group<RB>; a run-time one for the grouped decode kernel).
__device__ __forceinline__ bool resolve_group_rows(const W4Args& p, int y, int rb, int& e, int& m0, int& m_end) {
    const int lane = threadIdx.x & 63;
    int base = 0;  // row blocks of the groups before this step's
    for (int e0 = 0; e0 < p.num_groups; e0 += 64) {
        const int g = e0 + lane;
        int r0 = 0, r1 = 0;
        if (g < p.num_groups) {
            r0 = min(max(p.offsets[g], 0), p.row_capacity);
            r1 = min(max(p.offsets[g + 1], r0), p.row_capacity);
        }
        const int nb = (r1 - r0 + rb - 1) / rb;
        int incl = nb;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int v = __shfl_up(incl, d, 64);
            if (lane >= d) incl += v;
        }
        const int excl = incl - nb;
        const uint64_t hit = __ballot(y >= base + excl && y < base + incl);
        if (hit) {
            const int src = __builtin_ctzll(hit);
            e = __builtin_amdgcn_readfirstlane(e0 + src);
            m0 = __builtin_amdgcn_readfirstlane(__shfl(r0, src, 64) + rb * (y - base - __shfl(excl, src, 64)));
            m_end = __builtin_amdgcn_readfirstlane(__shfl(r1, src, 64));
            return true;
        }
        base += __shfl(incl, 63, 64);
    }
    return false;
}
template <int RB = 16>
__device__ __forceinline__ bool resolve_group(const W4Args& p, int y, int& e, int& m0, int& m_end) {
    return resolve_group_rows(p, y, RB, e, m0, m_end);
}

// Eight activations (row `off / K`, k = off % K .. +7) as bf16 MFMA operands.
template <bool F32A>
__device__ __forceinline__ void load_a8(const void* A, int64_t off, bool ok, u32x4_t& hi,
                                        u32x4_t& lo) {
    if (!ok) {
        hi = u32x4_t{0, 0, 0, 0};
        lo = u32x4_t{0, 0, 0, 0};
        return;
    }
    if constexpr (F32A) {
        const float4* p = reinterpret_cast<const float4*>(static_cast<const float*>(A) + off);
        const float4 x0 = p[0], x1 = p[1];
        const float v[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint16_t h0 = f32_to_bf16(v[2 * i]), h1 = f32_to_bf16(v[2 * i + 1]);
            hi[i] = static_cast<uint32_t>(h0) | (static_cast<uint32_t>(h1) << 16);
            lo[i] = pack_bf16x2(v[2 * i] - bf16_to_f32(h0), v[2 * i + 1] - bf16_to_f32(h1));
        }
    } else {
        hi = *reinterpret_cast<const u32x4_t*>(static_cast<const uint16_t*>(A) + off);
        lo = u32x4_t{0, 0, 0, 0};
    }
}

// Output element (row r, column c) of a W4 GEMM: fp32 with the reference's
// alpha / beta (beta == 0 never reads C, gemm_quant.cpp:12-21) or bf16 RNE.
template <bool F32C>
__device__ __forceinline__ void w4_store(const W4Args& p, int64_t o, float v) {
    if constexpr (F32C) {
        float* Cp = static_cast<float*>(p.C);
        float out = p.alpha * v;
        if (p.beta != 0.0f) out = p.beta * Cp[o] + out;
        Cp[o] = out;
    } else {
        static_cast<uint16_t*>(p.C)[o] = f32_to_bf16(v);
    }
}

// SwiGLU of one (gate, up) pair, moe.cpp:144-146 and :191: silu(g) * u with
// silu(v) = v / (1 + exp(-v)), fp32, IEEE division.
__device__ __forceinline__ float swiglu(float g, float u) { return g / (1.0f + expf(-g)) * u; }

// SwiGLU epilogue (SWI): the weights interleave the gate and up projections
// by column tile (lhq_w4_interleave_gate_up): tile 2j holds gate columns
// 16j .. 16j+15 and tile 2j+1 the same up columns, so the accumulators of
// one gate column and its up column sit in the same lane of two adjacent
// tiles.  The kernel then writes act[r][16j + c] = bf16(swiglu(g, u)) with
// p.N = the intermediate width (act's row length) and p.Nt = 2 ceil(N/16).

// A pointer that is the same in every lane, moved to scalar registers.
template <typename T>
__device__ __forceinline__ T* uniform_ptr(T* q) {
    const uint64_t v = reinterpret_cast<uint64_t>(q);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(v >> 32));
    return reinterpret_cast<T*>((static_cast<uint64_t>(hi) << 32) | lo);
}

// word 3 of a raw buffer resource (gfx9 family): 32-bit data format, no
// swizzle, offsets taken as given
constexpr int kBufWord3 = 0x00020000;
#define LHQ_LDS_AS __attribute__((address_space(3)))

// w4stream.hip: a few rows of a plain call against streamed weights (bf16 or
// the fp32 interface).  w4_stream_rb: its 16-row blocks per workgroup for
// this call, 0 where it is not the choice.
int w4_stream_rb(const W4Args& a, bool f32);
int launch_w4_stream(const W4Args& a, bool f32, int rb, hipStream_t s, const char* who);
int w4_device_cus();

}  // namespace lhq
