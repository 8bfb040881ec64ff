// quant.hip -- int8 / int4 / fp8 quantizers and dequantizers for gfx950,
// bit-exact with the reference (quant.cpp:12-249).
//
// Bit-exactness rests on three facts the kernels respect:
//   * max|x| is order-independent (the reference's `a > m` never lets NaN
//     win, quant.cpp:21-28; the kernels use the same compare-and-select), so
//     any reduction tree gives the reference's maximum;
//   * the scale uses the same IEEE operations: m / 127 (or /7, /448) and
//     1 / scale are correctly rounded divisions in HIP device code;
//   * rounding is saturate-then-round-to-nearest-even (quant.cpp:12-19), with
//     per-row / per-tensor multiplying by the reciprocal and per-column /
//     int4 group dividing by the scale, exactly as the reference does.
//   * no multiply-add is fused anywhere in this file.
#include "common.hpp"

#include <algorithm>

#pragma clang fp contract(off)

namespace lhq {
namespace {

constexpr int kBlock = 256;

// max(m, a) in the reference's form `if (a > m) m = a` (quant.cpp:21-28):
// a NaN `a` never replaces m, whatever kind of NaN it is.
__device__ __forceinline__ float amax(float m, float a) { return (a > m) ? a : m; }

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v = amax(v, __shfl_xor(v, off, 64));
    return v;
}

// Block-wide max of non-negative values (NaN never wins); result broadcast.
__device__ float block_max(float v) {
    __shared__ float part[kBlock / 64];
    v = wave_max(v);
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    if (lane == 0) part[w] = v;
    __syncthreads();
    float r = part[0];
#pragma unroll
    for (int i = 1; i < kBlock / 64; ++i) r = amax(r, part[i]);
    __syncthreads();
    return r;
}

template <typename T> __device__ __forceinline__ float load_f(const T* p, int64_t i);
template <> __device__ __forceinline__ float load_f<float>(const float* p, int64_t i) { return p[i]; }
template <> __device__ __forceinline__ float load_f<uint16_t>(const uint16_t* p, int64_t i) {
    return bf16_to_f32(p[i]);
}

// log2 of the threads that a workgroup gives the four-column words of a row.
inline int column_bits(int64_t quads) {
    int cb = 0;
    while (cb < 8 && (int64_t{1} << cb) < quads) ++cb;
    return cb;
}

// Quantize one value with a reciprocal (per-row / per-tensor) -- int8 or fp8.
template <bool FP8>
__device__ __forceinline__ uint8_t quant_mul(float x, float inv) {
    if constexpr (FP8) return f32_to_e4m3(x * inv);
    else return static_cast<uint8_t>(static_cast<int8_t>(sat_rint(x * inv, 127)));
}
// Four values with a reciprocal, as one word (value j in byte j).
template <bool FP8>
__device__ __forceinline__ uint32_t quant_mul4(float a, float b, float c, float d, float inv) {
    if constexpr (FP8) {
        return pack_e4m3x2(a * inv, b * inv) | (pack_e4m3x2(c * inv, d * inv) << 16);
    } else {
        auto q = [inv](float x) { return static_cast<uint32_t>(sat_rint(x * inv, 127)) & 0xffu; };
        return q(a) | (q(b) << 8) | (q(c) << 16) | (q(d) << 24);
    }
}

// rint(x / s) of a finite quotient below 256 in magnitude without the IEEE
// division (about ten instructions an element): r = x * rs with rs = rcp(s)
// (1 ulp) is within 256 * 2^-22 of x / s, and the correctly rounded quotient
// within 256 * 2^-24 of it, so where r lies more than 2^-13 from a
// half-integer both round to the same integer.  False (about 1 value in 4000,
// and every NaN, infinite or larger quotient): the caller divides.
__device__ __forceinline__ bool rint_quotient(float x, float rs, float& t) {
    const float r = x * rs;
    t = __builtin_rintf(r);
    return fabsf(r) < 256.0f && fabsf(fabsf(r - t) - 0.5f) > 0x1p-13f;
}

// One workgroup per row: max-abs, scale = m / QMAX (1 if m == 0),
// inv = 1 / scale, q = round(x * inv)  (quant.cpp:52-63, 195-206).
template <typename T, bool FP8>
__global__ __launch_bounds__(kBlock) void quant_per_row_kernel(const T* __restrict__ src,
                                                               uint8_t* __restrict__ dst,
                                                               float* __restrict__ scales, int dim) {
    const int64_t base = static_cast<int64_t>(blockIdx.x) * dim;
    float m = 0.0f;
    for (int i = threadIdx.x; i < dim; i += kBlock) m = amax(m, fabsf(load_f(src, base + i)));
    m = block_max(m);
    const float qmax = FP8 ? 448.0f : 127.0f;
    const float scale = (m > 0.0f) ? m / qmax : 1.0f;
    const float inv = 1.0f / scale;
    for (int i = threadIdx.x; i < dim; i += kBlock) dst[base + i] = quant_mul<FP8>(load_f(src, base + i), inv);
    if (threadIdx.x == 0) scales[blockIdx.x] = scale;
}

// fp32 rows whose length is a multiple of 4: 16-byte loads and 4-byte
// stores; rows of up to R * 4 * kBlock elements stay in registers between
// the max-abs pass and the quantizing pass (one read of the row), longer
// rows are read again (from L2).  Same rule as quant_per_row_kernel.
// R (16-byte chunks a thread keeps) is the least of 1, 2, 4, 8 that holds a
// row (int8, 512 rows of 1024 2.6 us, 4096 of 512 5.3; eight for all 3.1, 6.8).
template <bool FP8, int R>
__global__ __launch_bounds__(kBlock) void quant_per_row_f32_vec_kernel(const float* __restrict__ src,
                                                                       uint8_t* __restrict__ dst,
                                                                       float* __restrict__ scales, int dim) {
    const int64_t base = static_cast<int64_t>(blockIdx.x) * dim;
    const f32x4_t* s4 = reinterpret_cast<const f32x4_t*>(src + base);
    const int n4 = dim >> 2;
    const bool cached = n4 <= R * kBlock;
    f32x4_t keep[R];
    float m = 0.0f;
    if (cached) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int i = threadIdx.x + r * kBlock;
            keep[r] = i < n4 ? s4[i] : f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < 4; ++j) m = amax(m, fabsf(keep[r][j]));
        }
    } else {
        for (int i = threadIdx.x; i < n4; i += kBlock) {
            const f32x4_t v = s4[i];
#pragma unroll
            for (int j = 0; j < 4; ++j) m = amax(m, fabsf(v[j]));
        }
    }
    m = block_max(m);
    const float qmax = FP8 ? 448.0f : 127.0f;
    const float scale = (m > 0.0f) ? m / qmax : 1.0f;
    const float inv = 1.0f / scale;
    uint32_t* d4 = reinterpret_cast<uint32_t*>(dst + base);
    auto put = [&](int i, const f32x4_t& v) {
        d4[i] = quant_mul4<FP8>(v[0], v[1], v[2], v[3], inv);
    };
    if (cached) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int i = threadIdx.x + r * kBlock;
            if (i < n4) put(i, keep[r]);
        }
    } else {
        for (int i = threadIdx.x; i < n4; i += kBlock) put(i, s4[i]);
    }
    if (threadIdx.x == 0) scales[blockIdx.x] = scale;
}

// bf16 rows whose length is a multiple of 8: 16-byte loads, 8-byte stores;
// rows of up to R * 8 * kBlock elements stay in registers between the two
// passes, longer rows are read again (from L2).  Bound by memory: 2048 rows
// of 4096 move 25 MB in 7.4 us at best (9.6 with a second read of the row).
// R (16-byte chunks a thread keeps) is the least of 1, 2, 4, 8 that holds a row
// (16 rows of 14336 5.6 us; four and a second read 6.7).
template <bool FP8, int R>
__global__ __launch_bounds__(kBlock) void quant_per_row_bf16_vec_kernel(const uint16_t* __restrict__ src,
                                                                        uint8_t* __restrict__ dst,
                                                                        float* __restrict__ scales,
                                                                        int dim) {
    const int64_t base = static_cast<int64_t>(blockIdx.x) * dim;
    const u32x4_t* s4 = reinterpret_cast<const u32x4_t*>(src + base);
    const int n8 = dim >> 3;
    const bool cached = n8 <= R * kBlock;
    u32x4_t keep[R];
    float m = 0.0f;
    auto scan = [&](const u32x4_t& v) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            m = amax(m, fabsf(__uint_as_float(v[j] << 16)));
            m = amax(m, fabsf(__uint_as_float(v[j] & 0xffff0000u)));
        }
    };
    if (cached) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int i = threadIdx.x + r * kBlock;
            keep[r] = i < n8 ? s4[i] : u32x4_t{0, 0, 0, 0};
        }
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (threadIdx.x + r * kBlock < n8) scan(keep[r]);  // (idle waves skip it)
    } else {
        for (int i = threadIdx.x; i < n8; i += kBlock) scan(s4[i]);
    }
    m = block_max(m);
    const float qmax = FP8 ? 448.0f : 127.0f;
    const float scale = (m > 0.0f) ? m / qmax : 1.0f;
    const float inv = 1.0f / scale;
    u32x2_t* d2 = reinterpret_cast<u32x2_t*>(dst + base);
    auto put = [&](int i, const u32x4_t& v) {
        auto lo = [](uint32_t w) { return __uint_as_float(w << 16); };
        auto hi = [](uint32_t w) { return __uint_as_float(w & 0xffff0000u); };
        d2[i] = u32x2_t{quant_mul4<FP8>(lo(v[0]), hi(v[0]), lo(v[1]), hi(v[1]), inv),
                        quant_mul4<FP8>(lo(v[2]), hi(v[2]), lo(v[3]), hi(v[3]), inv)};
    };
    if (cached) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int i = threadIdx.x + r * kBlock;
            if (i < n8) put(i, keep[r]);
        }
    } else {
        for (int i = threadIdx.x; i < n8; i += kBlock) put(i, s4[i]);
    }
    if (threadIdx.x == 0) scales[blockIdx.x] = scale;
}

// Per-column scales (quant.cpp:75-96, 218-238), in three launches that need
// no scratch memory of their own:
//   (1) a grid of (256 columns) x (row chunk) workgroups: each wave reduces
//       a quarter of the chunk's rows, four adjacent columns per lane with
//       16-byte loads, the waves meet in LDS, and the chunk's maxima go to
//       dst, chunk i's at bytes [4 i cols, 4 (i + 1) cols) -- chunks are at
//       least 64 rows (or all of them), so they fit, and (3) overwrites them -- or, where one
//       chunk holds all rows (dst may then be smaller), to the scales array.
//       Maxima are order-independent and NaN never wins, so any split gives
//       the reference's;
//   (2) the maximum over the chunks, as the scale m / QMAX (1 where m == 0);
//   (3) quantize: a thread takes its four columns' scales (and reciprocals)
//       once and walks R rows (8, or 2 up to 2^18 words of the matrix); a
//       workgroup spans 4 << cb columns, all 1024 or the least power of two
//       that holds a narrower matrix's, its other threads on further rows.
// Bound by memory: the fp32 matrix is read twice (the second time partly
// from the Infinity Cache) and the codes written.  K=4096, N=14336: 36 us
// for (1) and 46 for (3); N=4097: 15 and 22.  (A thread per four columns of
// a 64-row chunk with atomic maxima, and an IEEE division and a scale load
// per element, took 111 us and 55 us in all.)
// Any column count and 4-byte alignment; where a row's length is no multiple
// of four its last four columns are read and written as one word, some of them
// twice (column by column 16 rows of 255 took twice as long).  Rows of fewer
// than four columns are taken one by one.
__global__ __launch_bounds__(kBlock) void col_max_kernel(const float* __restrict__ src, uint8_t* __restrict__ maxw,
                                                         int rows, int cols, int chunk) {
    __shared__ float part[4][256];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c0 = blockIdx.x * 256 + lane * 4;
    const int cnt = min(4, cols - c0);  // <= 0 past the last column
    const int w0 = cols >= 4 ? min(c0, cols - 4) : c0;  // the four columns read
    const int last = min(cnt, 4) - 1;                   // (of fewer than four, the last one again)
    const int64_t chunks = (static_cast<int64_t>(rows) + chunk - 1) / chunk;
    // (the grid's y extent is capped, so very tall inputs give a workgroup several chunks)
    for (int64_t q = blockIdx.y; q < chunks; q += gridDim.y) {
        float m[4] = {0.f, 0.f, 0.f, 0.f};
        const int64_t r0 = q * chunk + wave * (chunk / 4);
        const int64_t r1 = min<int64_t>(rows, r0 + chunk / 4);
        // eight rows in flight; rows past the end read the last one again
        auto scan = [&](auto full) {
            for (int64_t r = r0; r < r1; r += 8) {
                f32x4_t v[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    const float* p = src + min(r + i, r1 - 1) * cols + w0;
                    if constexpr (full.value) v[i] = load_f32x4<true>(p, 4);
                    else v[i] = f32x4_t{p[0], p[min(1, last)], p[last], 0.f};
                }
#pragma unroll
                for (int i = 0; i < 8; ++i)
#pragma unroll
                    for (int j = 0; j < 4; ++j) m[j] = amax(m[j], fabsf(v[i][j]));
            }
        };
        if (cols >= 4) scan(Full{});
        else if (cnt > 0) scan(Part{});
        __syncthreads();
        if (w0 == c0) {
            *reinterpret_cast<f32x4_t*>(&part[wave][lane * 4]) = f32x4_t{m[0], m[1], m[2], m[3]};
        } else {
#pragma unroll
            for (int j = 1; j < 4; ++j)
                if (j >= c0 - w0) part[wave][lane * 4 + j - (c0 - w0)] = m[j];
        }
        __syncthreads();
        const int c = blockIdx.x * 256 + static_cast<int>(threadIdx.x);
        float t = part[0][threadIdx.x];
#pragma unroll
        for (int w = 1; w < 4; ++w) t = amax(t, part[w][threadIdx.x]);
        if (c < cols) __builtin_memcpy(maxw + 4 * (q * cols + c), &t, 4);
    }
}

// A workgroup takes 64 columns, its waves every fourth chunk, four loads in
// flight.  scales may be maxw itself (one chunk): a column's words are read
// by its own workgroup, before it writes the scale.
template <bool FP8>
__global__ __launch_bounds__(kBlock) void col_scale_kernel(const uint8_t* maxw, int chunks, float* scales, int cols) {
    __shared__ float part[4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = blockIdx.x * 64 + lane;
    const int cc = min(c, cols - 1);
    float m = 0.0f;
    for (int q = wave; q < chunks; q += 16) {
        float t[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)  // past the last chunk: the last one again
            __builtin_memcpy(&t[u], maxw + 4 * (static_cast<int64_t>(min(q + 4 * u, chunks - 1)) * cols + cc), 4);
#pragma unroll
        for (int u = 0; u < 4; ++u) m = amax(m, t[u]);
    }
    part[wave][lane] = m;
    __syncthreads();
    if (wave != 0 || c >= cols) return;
#pragma unroll
    for (int w = 1; w < 4; ++w) m = amax(m, part[w][lane]);
    const float qmax = FP8 ? 448.0f : 127.0f;
    scales[c] = (m > 0.0f) ? m / qmax : 1.0f;
}

// q = round(x / scale[c]).
template <bool FP8, int R>
__global__ __launch_bounds__(kBlock) void quant_per_col_kernel(const float* __restrict__ src,
                                                               const float* __restrict__ scales,
                                                               uint8_t* __restrict__ dst, int rows, int cols,
                                                               int cb) {
    const int c0 = static_cast<int>(((blockIdx.x << cb) + (threadIdx.x & ((1u << cb) - 1))) * 4);
    if (c0 >= cols) return;
    const int sub = kBlock >> cb;  // row groups of a workgroup
    const int cnt = min(4, cols - c0);
    const int w0 = cols >= 4 ? min(c0, cols - 4) : c0;  // a ragged row's last word overlaps the one before
    auto body = [&](auto full) {
        const f32x4_t sc = load_f32x4<full.value>(scales + w0, cnt);
        f32x4_t rs;
#pragma unroll
        for (int j = 0; j < 4; ++j) rs[j] = __builtin_amdgcn_rcpf(sc[j]);
        for (int64_t r0 = (static_cast<int64_t>(blockIdx.y) * sub + (threadIdx.x >> cb)) * R; r0 < rows;
             r0 += static_cast<int64_t>(gridDim.y) * sub * R) {
            const int64_t left = rows - r0;
            f32x4_t v[R];
#pragma unroll
            for (int i = 0; i < R; ++i) {
                const float* p = src + (r0 + min<int64_t>(i, left - 1)) * cols + w0;
                if constexpr (full.value) v[i] = load_f32x4<true>(p, 4);
                else v[i] = f32x4_t{p[0], p[min(1, cnt - 1)], p[cnt - 1], 0.f};
            }
#pragma unroll
            for (int i = 0; i < R; ++i) {
                if (i >= left) break;
                uint32_t o = 0;
                if constexpr (FP8) {
                    o = pack_e4m3x2(v[i][0] / sc[0], v[i][1] / sc[1]) |
                        (pack_e4m3x2(v[i][2] / sc[2], v[i][3] / sc[3]) << 16);
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        float t;
                        if (!rint_quotient(v[i][j], rs[j], t)) t = __builtin_rintf(v[i][j] / sc[j]);
                        o |= (static_cast<uint32_t>(sat_rint(t, 127)) & 0xffu) << (8 * j);
                    }
                }
                store_u8x4<full.value>(dst + (r0 + i) * cols + w0, o, cnt);
            }
        }
    };
    if (cols >= 4) body(Full{});
    else body(Part{});
}

// Per-tensor, up to kSmallTensor elements (the activations of a decode
// batch): one launch.  Every workgroup takes the maximum over the whole
// tensor (from L2) and quantizes its own kSmallSlice elements; the first one
// writes the scale.  24 x 4096 values: 6.1 us, where four launches (clear,
// atomic max, quantize, finalize) took 10.4 us of kernels and their gaps.
// The repeated reads grow with the size: 7.2 us at 2^17 values, where the
// three launches below take 2.6 + 1.6 + 3.4 and two gaps.
constexpr int kSmallThreads = 1024;
constexpr int kSmallSlice = 4 * kSmallThreads;
constexpr int64_t kSmallTensor = int64_t{1} << 17;

template <bool FP8>
__device__ __forceinline__ float tensor_scale(float m) {
    return (m > 0.0f) ? m / (FP8 ? 448.0f : 127.0f) : 1.0f;
}

template <bool FP8>
__global__ __launch_bounds__(kSmallThreads) void quant_tensor_small_kernel(const float* __restrict__ src,
                                                                           uint8_t* __restrict__ dst, int n,
                                                                           float* __restrict__ scale_out) {
    __shared__ float part[kSmallThreads / 64];
    const int mine = static_cast<int>(blockIdx.x) * kSmallSlice + 4 * static_cast<int>(threadIdx.x);
    f32x4_t x = {0.f, 0.f, 0.f, 0.f};
    if (mine + 4 <= n) x = load_f32x4<true>(src + mine, 4);
    else if (mine < n) x = load_f32x4<false>(src + mine, n - mine);
    float m = 0.0f;
    auto scan = [&m](const f32x4_t& v) {
#pragma unroll
        for (int j = 0; j < 4; ++j) m = amax(m, fabsf(v[j]));
    };
    const int n4 = n & ~3;
    int i = 4 * static_cast<int>(threadIdx.x);
    for (; i + 7 * kSmallSlice < n4; i += 8 * kSmallSlice) {  // eight loads in flight
        f32x4_t v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = load_f32x4<true>(src + i + u * kSmallSlice, 4);
#pragma unroll
        for (int u = 0; u < 8; ++u) scan(v[u]);
    }
    for (; i < n4; i += kSmallSlice) scan(load_f32x4<true>(src + i, 4));
    if (static_cast<int>(threadIdx.x) < n - n4) m = amax(m, fabsf(src[n4 + threadIdx.x]));
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    m = part[0];
#pragma unroll
    for (int w = 1; w < kSmallThreads / 64; ++w) m = amax(m, part[w]);
    const float scale = tensor_scale<FP8>(m);
    const uint32_t w = quant_mul4<FP8>(x[0], x[1], x[2], x[3], 1.0f / scale);
    if (mine + 4 <= n) store_u8x4<true>(dst + mine, w, 4);
    else if (mine < n) store_u8x4<false>(dst + mine, w, n - mine);
    if (blockIdx.x == 0 && threadIdx.x == 0) *scale_out = scale;
}

// Per-tensor, larger: (1) up to kMaxParts workgroups each put the maximum of
// their grid-stride share in a word of dst (which has n > 4 kMaxParts bytes
// and is overwritten by (3); no shared atomic), (2) one workgroup turns them
// into the scale, (3) quantize with the reciprocal.  Bound by memory, the
// tensor read twice: 4096 x 14336 fp32 96 us a call (with an atomic maximum
// per workgroup, single loads and a software e4m3 conversion 153 us for int8
// and 182 for fp8), 2048 x 4096 17 us (49).
constexpr int kMaxParts = 2048;

__global__ __launch_bounds__(kBlock) void tensor_max_kernel(const float* __restrict__ src, int64_t n,
                                                            uint8_t* __restrict__ parts) {
    float m = 0.0f;
    auto scan = [&m](const f32x4_t& v) {
#pragma unroll
        for (int j = 0; j < 4; ++j) m = amax(m, fabsf(v[j]));
    };
    const int64_t step = static_cast<int64_t>(gridDim.x) * kBlock * 4, n4 = n & ~int64_t{3};
    int64_t i = (static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x) * 4;
    for (; i + 3 * step < n4; i += 4 * step) {
        f32x4_t v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = load_f32x4<true>(src + i + u * step, 4);
#pragma unroll
        for (int u = 0; u < 4; ++u) scan(v[u]);
    }
    for (; i < n4; i += step) scan(load_f32x4<true>(src + i, 4));
    if (blockIdx.x == 0 && threadIdx.x < n - n4) m = amax(m, fabsf(src[n4 + threadIdx.x]));
    m = block_max(m);
    if (threadIdx.x == 0) __builtin_memcpy(parts + 4 * static_cast<int64_t>(blockIdx.x), &m, 4);
}

template <bool FP8>
__global__ __launch_bounds__(kBlock) void tensor_scale_kernel(const uint8_t* __restrict__ parts, int count,
                                                              float* __restrict__ scale_out) {
    float m = 0.0f;
    for (int i = threadIdx.x; i < count; i += kBlock) {
        float p;
        __builtin_memcpy(&p, parts + 4 * static_cast<int64_t>(i), 4);
        m = amax(m, p);
    }
    m = block_max(m);
    if (threadIdx.x == 0) *scale_out = tensor_scale<FP8>(m);
}

template <bool FP8>
__global__ __launch_bounds__(kBlock) void quant_tensor_kernel(const float* __restrict__ src,
                                                              uint8_t* __restrict__ dst, int64_t n,
                                                              const float* __restrict__ scale) {
    const float inv = 1.0f / *scale;
    const int64_t step = static_cast<int64_t>(gridDim.x) * kBlock * 4;
    int64_t i = (static_cast<int64_t>(blockIdx.x) * kBlock + threadIdx.x) * 4;
    for (; i + 3 * step + 4 <= n; i += 4 * step) {
        f32x4_t v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = load_f32x4<true>(src + i + u * step, 4);
#pragma unroll
        for (int u = 0; u < 4; ++u)
            store_u8x4<true>(dst + i + u * step, quant_mul4<FP8>(v[u][0], v[u][1], v[u][2], v[u][3], inv), 4);
    }
    for (; i < n; i += step) {
        const int cnt = static_cast<int>(min<int64_t>(4, n - i));
        const f32x4_t v = load_f32x4<false>(src + i, cnt);
        store_u8x4<false>(dst + i, quant_mul4<FP8>(v[0], v[1], v[2], v[3], inv), cnt);
    }
}

// n = 0: the scale of an empty tensor.
__global__ void unit_scale_kernel(float* w) { *w = 1.0f; }

// Dequantizers: dst = decode(src) * scale (quant.cpp:47-50, 65-73, 98-105,
// 190-193, 208-216, 240-249); MODE 0 = per-tensor, 1 = per-row, 2 = per-col.
template <bool FP8, int MODE>
__global__ void dequant_kernel(const uint8_t* __restrict__ src, const float* __restrict__ scales,
                               float* __restrict__ dst, int dim, int64_t n) {
    const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float s = (MODE == 0) ? scales[0] : (MODE == 1) ? scales[i / dim] : scales[i % dim];
    const float v = FP8 ? e4m3_to_f32(src[i]) : static_cast<float>(static_cast<int8_t>(src[i]));
    dst[i] = v * s;
}

// int4 symmetric, reference layout.  Scales: a thread per (group, column):
// m = max |w| over the group, s = m / 7 (1 if 0)  (quant.cpp:128-144).
__global__ void q4_scales_kernel(const float* __restrict__ src, float* __restrict__ scales, int N, int G,
                                 int64_t total) {
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const int n = static_cast<int>(t % N);
    const int64_t g = t / N;
    float m = 0.0f;
    for (int kk = 0; kk < G; ++kk) m = amax(m, fabsf(src[(g * G + kk) * N + n]));
    scales[t] = (m > 0.0f) ? m / 7.0f : 1.0f;
}

// Pack rows (2i, 2i+1) of column n into byte i*N + n, low nibble first; each
// row uses its own group's scale, division then saturating round to [-7, 7]
// (quant.cpp:146-159).
__global__ void q4_pack_kernel(const float* __restrict__ src, const float* __restrict__ scales,
                               uint8_t* __restrict__ packed, int N, int G, int64_t total) {
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const int n = static_cast<int>(t % N);
    const int64_t i = t / N;
    const int64_t k = 2 * i;
    const float s0 = scales[(k / G) * N + n];
    const float s1 = scales[((k + 1) / G) * N + n];
    const int q0 = sat_rint(src[k * N + n] / s0, 7);
    const int q1 = sat_rint(src[(k + 1) * N + n] / s1, 7);
    packed[t] = static_cast<uint8_t>((q0 & 0xf) | ((q1 & 0xf) << 4));
}

// Asymmetric int4 (no reference counterpart): per (group, column) the range
// is widened to contain 0, s = fp16((hi - lo) / 15) (1 if the range is empty,
// at least 2^-14), z = clamp(rint(-lo / s), 0, 15); codes
// u = clamp(rint(w / s) + z, 0, 15) use the fp16-rounded s.
__device__ __forceinline__ void q4a_params(float lo, float hi, uint16_t& sh_bits, float& sq, float& zf) {
    float s = (hi - lo) / 15.0f;
    if (!(s > 0.0f)) s = 1.0f;
    _Float16 sh = static_cast<_Float16>(s);  // RNE, like dtypes.hpp:17-55 for normal values
    sq = static_cast<float>(sh);
    if (sq < 0x1p-14f) {
        sh = static_cast<_Float16>(0x1p-14f);
        sq = 0x1p-14f;
    }
    zf = fminf(fmaxf(__builtin_rintf(-lo / sq), 0.0f), 15.0f);
    sh_bits = __builtin_bit_cast(uint16_t, sh);
}

__global__ void q4a_params_kernel(const float* __restrict__ src, uint16_t* __restrict__ scales,
                                  uint8_t* __restrict__ zeros, int N, int G, int64_t total) {
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const int n = static_cast<int>(t % N);
    const int64_t g = t / N;
    float lo = 0.0f, hi = 0.0f;
    for (int kk = 0; kk < G; ++kk) {
        const float w = src[(g * G + kk) * N + n];
        if (w < lo) lo = w;
        if (w > hi) hi = w;
    }
    float sq, zf;
    q4a_params(lo, hi, scales[t], sq, zf);
    zeros[t] = static_cast<uint8_t>(zf);
}

__global__ void q4a_pack_kernel(const float* __restrict__ src, const uint16_t* __restrict__ scales,
                                const uint8_t* __restrict__ zeros, uint8_t* __restrict__ packed, int N,
                                int G, int64_t total) {
    const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const int n = static_cast<int>(t % N);
    const int64_t i = t / N;
    uint32_t b = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int64_t k = 2 * i + h;
        const int64_t gi = (k / G) * N + n;
        const float sq = f16_to_f32(scales[gi]);
        float v = __builtin_rintf(src[k * N + n] / sq) + static_cast<float>(zeros[gi]);
        v = fminf(fmaxf(v, 0.0f), 15.0f);
        b |= static_cast<uint32_t>(v) << (4 * h);
    }
    packed[t] = static_cast<uint8_t>(b);
}

// Dequantize int4: a thread owns four adjacent columns and P packed rows,
// reading a 32-bit word of codes and writing two 16-byte runs of fp32 per
// packed row.  Bound by the write: K=4096, N=14336, G=128 writes 235 MB in 44
// us (a thread per element with two 64-bit divisions took 117).
// P is 4, and 1 up to 2^18 words of codes, where four rows a thread took 1.1
// to 1.5 times as long in the mean (K=64, N=8192 3.15 us, one row 2.19; K=2048,
// N=8192 one row 13.5, four 14.1 or as little as 0.82 of one).
// A workgroup spans 4 << cb columns: all 1024, or for narrower weights the
// least power of two that holds them, its other threads on further rows.
// Where N is no multiple of four a row's last four columns are one word too,
// some of them written twice (K=1024, N=411 2.2 us; 5.6 one by one); fewer than
// four columns are taken one by one.
template <bool ASYM, int P>
__global__ __launch_bounds__(kBlock) void q4_dequant_kernel(const uint8_t* __restrict__ packed,
                                                            const void* __restrict__ scales,
                                                            const uint8_t* __restrict__ zeros,
                                                            float* __restrict__ dst, int K, int N, int G, int cb) {
    const int c = static_cast<int>(((blockIdx.x << cb) + (threadIdx.x & ((1u << cb) - 1))) * 4);
    if (c >= N) return;
    const int cnt = min(4, N - c);
    const int c0 = N >= 4 ? min(c, N - 4) : c;
    const int sub = kBlock >> cb;  // row groups of a workgroup
    struct Params {
        f32x4_t s;
        uint32_t z;
    };
    auto body = [&](auto full) {
        constexpr bool F = full.value;
        auto params = [&](int g) {  // a group's scales and zero points
            const int64_t gi = static_cast<int64_t>(g) * N + c0;
            Params p = {{0.f, 0.f, 0.f, 0.f}, 0u};
            if constexpr (ASYM) {
                const uint16_t* sp = static_cast<const uint16_t*>(scales) + gi;
                if constexpr (F) {
                    uint16_t h[4];
                    __builtin_memcpy(h, sp, 8);
#pragma unroll
                    for (int j = 0; j < 4; ++j) p.s[j] = f16_to_f32(h[j]);
                } else {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (j < cnt) p.s[j] = f16_to_f32(sp[j]);
                }
                p.z = load_u8x4<F>(zeros + gi, cnt);
            } else {
                p.s = load_f32x4<F>(static_cast<const float*>(scales) + gi, cnt);
            }
            return p;
        };
        auto put = [&](int64_t k, uint32_t nib, const Params& p) {  // codes in the low nibbles of nib's bytes
            f32x4_t v;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int u = static_cast<int>((nib >> (8 * j)) & 0xfu);
                // sign extension, quant.hpp:73-74
                const int q = ASYM ? u - static_cast<int>((p.z >> (8 * j)) & 0xffu) : (u ^ 8) - 8;
                v[j] = static_cast<float>(q) * p.s[j];
            }
            store_f32x4<F>(dst + k * N + c0, v, cnt);
        };
        const int pairs = K / 2;
        for (int64_t i0 = (static_cast<int64_t>(blockIdx.y) * sub + (threadIdx.x >> cb)) * P; i0 < pairs;
             i0 += static_cast<int64_t>(gridDim.y) * sub * P) {
            uint32_t w[P];
            Params p[P];
#pragma unroll
            for (int u = 0; u < P; ++u) {
                const int64_t i = i0 + u < pairs ? i0 + u : pairs - 1;
                w[u] = load_u8x4<F>(packed + i * N + c0, cnt);
                p[u] = params(static_cast<int>(2 * i) / G);
            }
#pragma unroll
            for (int u = 0; u < P; ++u) {
                if (i0 + u >= pairs) break;
                const int k = static_cast<int>(2 * (i0 + u));
                put(k, w[u], p[u]);
                if (G % 2 != 0) p[u] = params((k + 1) / G);  // an odd group may end inside the pair
                put(k + 1, w[u] >> 4, p[u]);
            }
        }
    };
    if (N >= 4) body(Full{});
    else body(Part{});
}

template <bool ASYM>
void launch_q4_dequant(const uint8_t* packed, const void* scales, const uint8_t* zeros, float* dst, int K, int N,
                       int G, hipStream_t s) {
    const int64_t quads = ceil_div64(N, 4);
    const int cb = column_bits(quads);
    const int p = quads * (K / 2) > (1 << 18) ? 4 : 1;
    const dim3 grid(static_cast<unsigned>(ceil_div64(quads, int64_t{1} << cb)),
                    static_cast<unsigned>(min(ceil_div(K / 2, p * (kBlock >> cb)), 65535)));
    if (p == 4) q4_dequant_kernel<ASYM, 4><<<grid, kBlock, 0, s>>>(packed, scales, zeros, dst, K, N, G, cb);
    else q4_dequant_kernel<ASYM, 1><<<grid, kBlock, 0, s>>>(packed, scales, zeros, dst, K, N, G, cb);
}

// Groups of 32, 64, 128 or 256 rows, scales and codes in one pass over the
// weights: a workgroup owns 64 adjacent columns of one group, wave w its rows
// [w * R, (w + 1) * R) (G = 4 R), held in R registers per thread from one
// coalesced 256-byte load per row; the four waves' extrema meet in LDS, every
// thread then has its column's scale and writes the codes of its row pairs.
// Bound by the fp32 read: K=4096, N=14336, G=128 reads 235 MB and writes 30.
// (Two passes with a thread per column and per code byte, as the kernels
// below still do for other group sizes, took 165 us a call; this one 54, 4.9
// TB/s.  G = 32 / 64 / 256: 171 / 169 / 208 us before, 47 / 51 / 56 now.)
// Any N and any alignment: a lane reads and writes single elements.
template <bool ASYM, int R>
__global__ __launch_bounds__(256) void q4_group_kernel(const float* __restrict__ src, void* __restrict__ scales,
                                                       uint8_t* __restrict__ zeros, uint8_t* __restrict__ packed,
                                                       int N, int NG) {
    __shared__ float ext[2][4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n = blockIdx.x * 64 + lane;
    const int nc = min(n, N - 1);  // lanes past the last column read it again and write nothing
    for (int g = blockIdx.y; g < NG; g += gridDim.y) {
        const int64_t row0 = (static_cast<int64_t>(g) * 4 + wave) * R;
        const float* p = src + row0 * N + nc;
        float w[R];
#pragma unroll
        for (int r = 0; r < R; ++r) w[r] = p[static_cast<int64_t>(r) * N];
        // the same compare-and-select as a serial scan: NaN never wins
        float lo = 0.0f, hi = 0.0f;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            if constexpr (ASYM) {
                if (w[r] < lo) lo = w[r];
                if (w[r] > hi) hi = w[r];
            } else {
                hi = amax(hi, fabsf(w[r]));
            }
        }
        if constexpr (ASYM) ext[0][wave][lane] = lo;
        ext[1][wave][lane] = hi;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (ASYM) {
                const float l = ext[0][i][lane];
                if (l < lo) lo = l;
            }
            hi = amax(hi, ext[1][i][lane]);
        }
        __syncthreads();
        const int64_t gi = static_cast<int64_t>(g) * N + n;
        float s, z = 0.0f;
        if constexpr (ASYM) {
            uint16_t sh;
            q4a_params(lo, hi, sh, s, z);
            if (wave == 0 && n < N) {
                static_cast<uint16_t*>(scales)[gi] = sh;
                zeros[gi] = static_cast<uint8_t>(z);
            }
        } else {
            s = (hi > 0.0f) ? hi / 7.0f : 1.0f;
            if (wave == 0 && n < N) static_cast<float*>(scales)[gi] = s;
        }
        const float rs = __builtin_amdgcn_rcpf(s);
        auto code = [&](float x) -> uint32_t {
            float t;
            if (!rint_quotient(x, rs, t)) t = __builtin_rintf(x / s);
            if constexpr (ASYM) return static_cast<uint32_t>(fminf(fmaxf(t + z, 0.0f), 15.0f));
            else return static_cast<uint32_t>(sat_rint(t, 7)) & 0xfu;
        };
        uint8_t* q = packed + (row0 >> 1) * N + n;
        if (n < N) {
#pragma unroll
            for (int r = 0; r < R; r += 2)
                q[static_cast<int64_t>(r >> 1) * N] = static_cast<uint8_t>(code(w[r]) | (code(w[r + 1]) << 4));
        }
    }
}

template <bool ASYM>
bool launch_q4_group(const float* src, void* scales, uint8_t* zeros, uint8_t* packed, int K, int N, int G,
                     hipStream_t s) {
    const int NG = K / G;
    const dim3 grid(static_cast<unsigned>(ceil_div64(N, 64)), static_cast<unsigned>(min(NG, 65535)));
    if (G == 32) q4_group_kernel<ASYM, 8><<<grid, 256, 0, s>>>(src, scales, zeros, packed, N, NG);
    else if (G == 64) q4_group_kernel<ASYM, 16><<<grid, 256, 0, s>>>(src, scales, zeros, packed, N, NG);
    else if (G == 128) q4_group_kernel<ASYM, 32><<<grid, 256, 0, s>>>(src, scales, zeros, packed, N, NG);
    else if (G == 256) q4_group_kernel<ASYM, 64><<<grid, 256, 0, s>>>(src, scales, zeros, packed, N, NG);
    else return false;
    return true;
}

inline unsigned blocks_for(int64_t n, int bs = kBlock) { return static_cast<unsigned>(ceil_div64(n, bs)); }

template <bool FP8>
int quantize_per_tensor(const float* src, uint8_t* dst, float* scale_out, int64_t n, void* stream,
                        const char* who) {
    LHQ_REQUIRE(src && dst && scale_out, "%s: null pointer", who);
    LHQ_REQUIRE(n >= 0, "%s: negative n", who);
    hipStream_t s = as_stream(stream);
    if (n == 0) {
        unit_scale_kernel<<<1, 1, 0, s>>>(scale_out);
    } else if (n <= kSmallTensor) {
        quant_tensor_small_kernel<FP8><<<blocks_for(n, kSmallSlice), kSmallThreads, 0, s>>>(
            src, dst, static_cast<int>(n), scale_out);
    } else {
        const unsigned parts = static_cast<unsigned>(std::min<int64_t>(ceil_div64(n, 16 * kBlock), kMaxParts));
        tensor_max_kernel<<<parts, kBlock, 0, s>>>(src, n, dst);
        tensor_scale_kernel<FP8><<<1, kBlock, 0, s>>>(dst, static_cast<int>(parts), scale_out);
        const unsigned grid = static_cast<unsigned>(std::min<int64_t>(ceil_div64(n, 16 * kBlock), 1 << 20));
        quant_tensor_kernel<FP8><<<grid, kBlock, 0, s>>>(src, dst, n, scale_out);
    }
    return check_launch(who);
}

template <bool FP8, int MODE>
int dequantize(const uint8_t* src, const float* scales, float* dst, int64_t n, int dim, void* stream,
               const char* who) {
    LHQ_REQUIRE(src && scales && dst, "%s: null pointer", who);
    LHQ_REQUIRE(n >= 0 && (MODE == 0 || dim > 0 || n == 0), "%s: bad dims", who);
    if (n == 0) return LHQ_OK;
    dequant_kernel<FP8, MODE><<<blocks_for(n), kBlock, 0, as_stream(stream)>>>(src, scales, dst, dim, n);
    return check_launch(who);
}

template <typename T, bool FP8>
int quantize_per_row(const T* src, uint8_t* dst, float* scales, int rows, int dim, void* stream,
                     const char* who) {
    LHQ_REQUIRE(src && dst && scales, "%s: null pointer", who);
    LHQ_REQUIRE(rows >= 0 && dim >= 0, "%s: negative dims", who);
    if (rows == 0) return LHQ_OK;
    hipStream_t s = as_stream(stream);
    const bool vec = sizeof(T) == 2 && dim % 8 == 0 && (reinterpret_cast<uintptr_t>(src) & 15) == 0 &&
                     (reinterpret_cast<uintptr_t>(dst) & 7) == 0;
    if constexpr (sizeof(T) == 2) {
        if (vec) {
            if (dim <= 8 * kBlock) quant_per_row_bf16_vec_kernel<FP8, 1><<<rows, kBlock, 0, s>>>(src, dst, scales, dim);
            else if (dim <= 16 * kBlock)
                quant_per_row_bf16_vec_kernel<FP8, 2><<<rows, kBlock, 0, s>>>(src, dst, scales, dim);
            else if (dim <= 32 * kBlock)
                quant_per_row_bf16_vec_kernel<FP8, 4><<<rows, kBlock, 0, s>>>(src, dst, scales, dim);
            else quant_per_row_bf16_vec_kernel<FP8, 8><<<rows, kBlock, 0, s>>>(src, dst, scales, dim);
            return check_launch(who);
        }
    } else {
        if (dim % 4 == 0 && (reinterpret_cast<uintptr_t>(src) & 15) == 0 &&
            (reinterpret_cast<uintptr_t>(dst) & 3) == 0) {
            if (dim <= 4 * kBlock) quant_per_row_f32_vec_kernel<FP8, 1><<<rows, kBlock, 0, s>>>(src, dst, scales, dim);
            else if (dim <= 8 * kBlock)
                quant_per_row_f32_vec_kernel<FP8, 2><<<rows, kBlock, 0, s>>>(src, dst, scales, dim);
            else if (dim <= 16 * kBlock)
                quant_per_row_f32_vec_kernel<FP8, 4><<<rows, kBlock, 0, s>>>(src, dst, scales, dim);
            else quant_per_row_f32_vec_kernel<FP8, 8><<<rows, kBlock, 0, s>>>(src, dst, scales, dim);
            return check_launch(who);
        }
    }
    quant_per_row_kernel<T, FP8><<<rows, kBlock, 0, s>>>(src, dst, scales, dim);
    return check_launch(who);
}

template <bool FP8>
int quantize_per_col(const float* src, uint8_t* dst, float* scales, int rows, int cols, void* stream,
                     const char* who) {
    LHQ_REQUIRE(src && dst && scales, "%s: null pointer", who);
    LHQ_REQUIRE(rows >= 0 && cols >= 0, "%s: negative dims", who);
    if (cols == 0) return LHQ_OK;
    hipStream_t s = as_stream(stream);
    // long chunks (little to merge) where they still make four workgroups per CU
    const int64_t strips = ceil_div64(cols, 256);
    const int chunk = rows < 64                                ? max(4, ceil_div(rows, 4) * 4)
                      : strips * ceil_div64(rows, 256) >= 1024 ? 256
                      : strips * ceil_div64(rows, 128) >= 1024 ? 128
                                                             : 64;
    const int chunks = static_cast<int>(ceil_div64(rows, chunk));
    uint8_t* const maxw = chunks > 1 ? dst : reinterpret_cast<uint8_t*>(scales);
    if (rows > 0)
        col_max_kernel<<<dim3(static_cast<unsigned>(strips), static_cast<unsigned>(min(chunks, 65535))), kBlock, 0, s>>>(
            src, maxw, rows, cols, chunk);
    col_scale_kernel<FP8><<<blocks_for(cols, 64), kBlock, 0, s>>>(maxw, chunks, scales, cols);
    if (rows > 0) {
        const int64_t quads = ceil_div64(cols, 4);
        const int cb = column_bits(quads);
        const int r = quads * rows > (1 << 18) ? 8 : 2;
        const dim3 grid(static_cast<unsigned>(ceil_div64(quads, int64_t{1} << cb)),
                        static_cast<unsigned>(std::min<int64_t>(ceil_div64(rows, r * (kBlock >> cb)), 65535)));
        if (r == 8) quant_per_col_kernel<FP8, 8><<<grid, kBlock, 0, s>>>(src, scales, dst, rows, cols, cb);
        else quant_per_col_kernel<FP8, 2><<<grid, kBlock, 0, s>>>(src, scales, dst, rows, cols, cb);
    }
    return check_launch(who);
}

bool q4_dims_ok(int K, int N, int G) { return K > 0 && N > 0 && G > 0 && K % G == 0 && K % 2 == 0; }

}  // namespace
}  // namespace lhq

using namespace lhq;

extern "C" {

int lhq_q8_quantize_per_tensor(const float* src, int8_t* dst, float* scale_out, int64_t n, void* stream) {
    return quantize_per_tensor<false>(src, reinterpret_cast<uint8_t*>(dst), scale_out, n, stream,
                                      "q8_quantize_per_tensor");
}
int lhq_q8_dequantize_per_tensor(const int8_t* src, const float* scale, float* dst, int64_t n, void* stream) {
    return dequantize<false, 0>(reinterpret_cast<const uint8_t*>(src), scale, dst, n, 1, stream,
                                "q8_dequantize_per_tensor");
}
int lhq_q8_quantize_per_row(const float* src, int8_t* dst, float* scales, int rows, int dim, void* stream) {
    return quantize_per_row<float, false>(src, reinterpret_cast<uint8_t*>(dst), scales, rows, dim, stream,
                                          "q8_quantize_per_row");
}
int lhq_q8_quantize_per_row_bf16(const uint16_t* src, int8_t* dst, float* scales, int rows, int dim,
                                 void* stream) {
    return quantize_per_row<uint16_t, false>(src, reinterpret_cast<uint8_t*>(dst), scales, rows, dim, stream,
                                             "q8_quantize_per_row_bf16");
}
int lhq_q8_dequantize_per_row(const int8_t* src, const float* scales, float* dst, int rows, int dim,
                              void* stream) {
    LHQ_REQUIRE(rows >= 0 && dim >= 0, "q8_dequantize_per_row: negative dims");
    return dequantize<false, 1>(reinterpret_cast<const uint8_t*>(src), scales, dst,
                                static_cast<int64_t>(rows) * dim, dim, stream, "q8_dequantize_per_row");
}
int lhq_q8_quantize_per_col(const float* src, int8_t* dst, float* scales, int rows, int cols, void* stream) {
    return quantize_per_col<false>(src, reinterpret_cast<uint8_t*>(dst), scales, rows, cols, stream,
                                   "q8_quantize_per_col");
}
int lhq_q8_dequantize_per_col(const int8_t* src, const float* scales, float* dst, int rows, int cols,
                              void* stream) {
    LHQ_REQUIRE(rows >= 0 && cols >= 0, "q8_dequantize_per_col: negative dims");
    return dequantize<false, 2>(reinterpret_cast<const uint8_t*>(src), scales, dst,
                                static_cast<int64_t>(rows) * cols, cols, stream, "q8_dequantize_per_col");
}

int lhq_fp8_quantize_per_tensor(const float* src, uint8_t* dst, float* scale_out, int64_t n, void* stream) {
    return quantize_per_tensor<true>(src, dst, scale_out, n, stream, "fp8_quantize_per_tensor");
}
int lhq_fp8_dequantize_per_tensor(const uint8_t* src, const float* scale, float* dst, int64_t n,
                                  void* stream) {
    return dequantize<true, 0>(src, scale, dst, n, 1, stream, "fp8_dequantize_per_tensor");
}
int lhq_fp8_quantize_per_row(const float* src, uint8_t* dst, float* scales, int rows, int dim, void* stream) {
    return quantize_per_row<float, true>(src, dst, scales, rows, dim, stream, "fp8_quantize_per_row");
}
int lhq_fp8_dequantize_per_row(const uint8_t* src, const float* scales, float* dst, int rows, int dim,
                               void* stream) {
    LHQ_REQUIRE(rows >= 0 && dim >= 0, "fp8_dequantize_per_row: negative dims");
    return dequantize<true, 1>(src, scales, dst, static_cast<int64_t>(rows) * dim, dim, stream,
                               "fp8_dequantize_per_row");
}
int lhq_fp8_quantize_per_col(const float* src, uint8_t* dst, float* scales, int rows, int cols, void* stream) {
    return quantize_per_col<true>(src, dst, scales, rows, cols, stream, "fp8_quantize_per_col");
}
int lhq_fp8_dequantize_per_col(const uint8_t* src, const float* scales, float* dst, int rows, int cols,
                               void* stream) {
    LHQ_REQUIRE(rows >= 0 && cols >= 0, "fp8_dequantize_per_col: negative dims");
    return dequantize<true, 2>(src, scales, dst, static_cast<int64_t>(rows) * cols, cols, stream,
                               "fp8_dequantize_per_col");
}

int lhq_q4_quantize_groupwise(const float* src, uint8_t* packed, float* scales, int K, int N, int G,
                              void* stream) {
    LHQ_REQUIRE(src && packed && scales, "q4_quantize_groupwise: null pointer");
    LHQ_REQUIRE(q4_dims_ok(K, N, G), "q4_quantize_groupwise: need K,N,G > 0, K even, G | K (K=%d N=%d G=%d)",
                K, N, G);
    hipStream_t s = as_stream(stream);
    if (launch_q4_group<false>(src, scales, nullptr, packed, K, N, G, s)) return check_launch("q4_quantize_groupwise");
    const int64_t ns = static_cast<int64_t>(K / G) * N, np = static_cast<int64_t>(K / 2) * N;
    q4_scales_kernel<<<blocks_for(ns), kBlock, 0, s>>>(src, scales, N, G, ns);
    q4_pack_kernel<<<blocks_for(np), kBlock, 0, s>>>(src, scales, packed, N, G, np);
    return check_launch("q4_quantize_groupwise");
}

int lhq_q4_dequantize_groupwise(const uint8_t* packed, const float* scales, float* dst, int K, int N, int G,
                                void* stream) {
    LHQ_REQUIRE(packed && scales && dst, "q4_dequantize_groupwise: null pointer");
    LHQ_REQUIRE(q4_dims_ok(K, N, G), "q4_dequantize_groupwise: bad dims (K=%d N=%d G=%d)", K, N, G);
    launch_q4_dequant<false>(packed, scales, nullptr, dst, K, N, G, as_stream(stream));
    return check_launch("q4_dequantize_groupwise");
}

int lhq_q4a_quantize_groupwise(const float* src, uint8_t* packed, uint16_t* scales, uint8_t* zeros, int K,
                               int N, int G, void* stream) {
    LHQ_REQUIRE(src && packed && scales && zeros, "q4a_quantize_groupwise: null pointer");
    LHQ_REQUIRE(q4_dims_ok(K, N, G), "q4a_quantize_groupwise: bad dims (K=%d N=%d G=%d)", K, N, G);
    hipStream_t s = as_stream(stream);
    if (launch_q4_group<true>(src, scales, zeros, packed, K, N, G, s)) return check_launch("q4a_quantize_groupwise");
    const int64_t ns = static_cast<int64_t>(K / G) * N, np = static_cast<int64_t>(K / 2) * N;
    q4a_params_kernel<<<blocks_for(ns), kBlock, 0, s>>>(src, scales, zeros, N, G, ns);
    q4a_pack_kernel<<<blocks_for(np), kBlock, 0, s>>>(src, scales, zeros, packed, N, G, np);
    return check_launch("q4a_quantize_groupwise");
}

int lhq_q4a_dequantize_groupwise(const uint8_t* packed, const uint16_t* scales, const uint8_t* zeros,
                                 float* dst, int K, int N, int G, void* stream) {
    LHQ_REQUIRE(packed && scales && zeros && dst, "q4a_dequantize_groupwise: null pointer");
    LHQ_REQUIRE(q4_dims_ok(K, N, G), "q4a_dequantize_groupwise: bad dims (K=%d N=%d G=%d)", K, N, G);
    launch_q4_dequant<true>(packed, scales, zeros, dst, K, N, G, as_stream(stream));
    return check_launch("q4a_dequantize_groupwise");
}

}  // extern "C"
