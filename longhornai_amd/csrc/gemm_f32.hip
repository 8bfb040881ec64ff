// gemm_f32.hip -- fp32 GEMM behind the gemm.hpp drop-in (gemm.hpp:13-29),
// the route of the W4A16 calls that the int4 kernels do not take (their
// weights dequantized first) and of non-finite activations.
//
// fp32 MFMA (32x32x2: fp32 operands, products and sums, 157 TFLOP/s).  The
// waves of a workgroup split K, not the tile, so a small output still fills
// the chip: 100 rows x 4096 columns are 256 workgroups of eight waves.  Each
// wave works alone (no barrier in the K loop): per stage of 32 k it loads its
// rows of A whole (128 contiguous bytes a row) and turns them to operand order
// through its own 4 KiB of LDS per 32 rows, and loads B, whose rows already
// are operands (32 adjacent columns of one k), straight into registers, the
// next stage in flight while one is multiplied.  (A loaded in operand order, a
// 32-byte piece of 32 rows at a time, fetched every line four times: M = 512
// took 265 us.)  The partial tiles meet in LDS in wave order, so results are
// deterministic; many short sums instead of one long one also halve the
// error.  K = N = 4096: M = 100 51 us, 66 TFLOP/s (the 64x64 VALU tile that
// walks all of K 550); M = 1 28 us, 2.4 TB/s of B (502); M = 512 175 us, 98
// TFLOP/s (584).  Short K on many outputs stays on that tile (valu_wins).
//
// Semantics follow gemm.cpp: lh::gemm applies beta first and never reads C
// when beta == 0 (gemm.cpp:60-68); lh::gemm_ref always reads C and returns
// alpha*acc + beta*C (gemm.cpp:5-16).  grid.z walks a uniform batch
// (gemm.cpp:59-67).
#include "common.hpp"

namespace lhq {
namespace {

constexpr int kStage = 32;  // k per stage
constexpr int kXcds = 8;

__device__ __forceinline__ f32x16_t mfma_f32_32x32x2(float a, float b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// MI x NI blocks of 32 x 32 per workgroup, KS waves splitting K.
template <bool REF, int MI, int NI, int KS>
__global__ __launch_bounds__(64 * KS) void gemm_f32_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                           float* __restrict__ C, int M, int N, int K, int mt,
                                                           float alpha, float beta) {
    __shared__ __attribute__((aligned(16))) float red[KS][MI * NI * 16 * 64];
    const int64_t z = blockIdx.z;
    A += z * M * static_cast<int64_t>(K);
    B += z * K * static_cast<int64_t>(N);
    C += z * M * static_cast<int64_t>(N);
    // workgroups are dealt to the XCDs round-robin: the row tiles of one
    // column strip go to one XCD, whose L2 then reads the strip's B once; the
    // strips past a multiple of eight follow in order
    const int whole_strips = (N + 32 * NI - 1) / (32 * NI) / kXcds * kXcds;
    const int turn = static_cast<int>(blockIdx.x) - mt * whole_strips;  // < 0: one of the whole eights
    const int id = turn < 0 ? static_cast<int>(blockIdx.x) / kXcds : turn;
    const int m0 = (id % mt) * 32 * MI;
    const int n0 = (turn < 0 ? (id / mt) * kXcds + static_cast<int>(blockIdx.x) % kXcds : whole_strips + id / mt) * 32 * NI;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l = lane & 31, h = lane >> 5;
    const int stages = (K + kStage - 1) / kStage;
    const int s0 = static_cast<int>(static_cast<int64_t>(stages) * wave / KS);
    const int s1 = static_cast<int>(static_cast<int64_t>(stages) * (wave + 1) / KS);

    // rows and columns past the end read the last ones; their outputs are not stored
    const int ar = lane >> 3, ac = lane & 7;  // loads: row 8 q + ar, k 4 ac .. + 3 of a stage
    const float* ap[MI][4];
    const float* bp[NI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q)
            ap[i][q] = A + static_cast<int64_t>(min(m0 + 32 * i + 8 * q + ar, M - 1)) * K + 4 * ac;
#pragma unroll
    for (int j = 0; j < NI; ++j) bp[j] = B + static_cast<int64_t>(4 * h) * N + min(n0 + 32 * j + l, N - 1);

    f32x16_t acc[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

    // step t of a stage covers k = 32 s + 8 t + 4 h + i: the k order inside a
    // step is the same for A and B, which is all an MFMA's k slots need
    struct Regs {
        f32x4_t a[MI][4];
        float b[NI][4][4];
    };
    auto load = [&](Regs& r, int s, auto full) {
        const int k0 = s * kStage;
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                if constexpr (full.value) {
                    r.a[i][q] = load_f32x4<true>(ap[i][q] + k0, 4);
                } else {
                    // k past the end reads the row's last element and becomes
                    // zero: loads under a condition would wait for each other
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int k = k0 + 4 * ac + e;
                        const float v = ap[i][q][min(k, K - 1) - 4 * ac];
                        r.a[i][q][e] = k < K ? v : 0.0f;
                    }
                }
            }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int k = k0 + 8 * t;
#pragma unroll
            for (int j = 0; j < NI; ++j)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int ku = full.value ? k + u : min(k + u, K - 1 - 4 * h);
                    const float v = bp[j][static_cast<int64_t>(ku) * N];
                    r.b[j][t][u] = full.value || k + u + 4 * h < K ? v : 0.0f;
                }
        }
    };
    // the wave's own LDS (its part of red): row r's k 4 c .. + 3 in slot c ^ (r & 7)
    float* const mine = red[wave];
    auto multiply = [&](const Regs& r) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<f32x4_t*>(mine + (32 * i + 8 * q + ar) * kStage + 4 * (ac ^ ar)) = r.a[i][q];
        // the rows were written by other lanes of this wave: LDS is in order
        // within a wave, the fences keep the compiler to it (0.2-0.3% over
        // 4,684 shapes)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        f32x4_t a[MI][4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < MI; ++i)
                a[i][t] = *reinterpret_cast<const f32x4_t*>(mine + (32 * i + l) * kStage + 4 * ((2 * t + h) ^ (l & 7)));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int i = 0; i < MI; ++i)
#pragma unroll
                    for (int j = 0; j < NI; ++j) acc[i][j] = mfma_f32_32x32x2(a[i][t][u], r.b[j][t][u], acc[i][j]);
    };
    // whole stages, the next one's loads in flight while one is multiplied
    // (past the end the last one is read again), then the partial one
    const int whole = min(s1, K / kStage);
    if (s0 < whole) {
        Regs r0, r1;
        load(r0, s0, Full{});
        int s = s0;
        for (; s + 2 <= whole; s += 2) {
            load(r1, s + 1, Full{});
            __builtin_amdgcn_sched_barrier(0);  // keeps the loads ahead of the products
            multiply(r0);
            load(r0, min(s + 2, whole - 1), Full{});
            __builtin_amdgcn_sched_barrier(0);
            multiply(r1);
        }
        if (s < whole) multiply(r0);
    }
    if (s1 > whole && s0 < s1) {
        Regs r;
        load(r, stages - 1, Part{});
        multiply(r);
    }

    // D element e of lane (h, l): row 8 (e / 4) + 4 h + e % 4, column l
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) red[wave][((i * NI + j) * 16 + e) * 64 + lane] = acc[i][j][e];
    __syncthreads();
    for (int x = threadIdx.x; x < MI * NI * 16 * 64; x += 64 * KS) {
        const int e = (x >> 6) & 15, ij = x >> 10;
        const int m = m0 + 32 * (ij / NI) + 8 * (e >> 2) + 4 * ((x >> 5) & 1) + (e & 3);
        const int n = n0 + 32 * (ij % NI) + (x & 31);
        float v = red[0][x];
#pragma unroll
        for (int w = 1; w < KS; ++w) v += red[w][x];
        if (m >= M || n >= N) continue;
        float* c = C + static_cast<int64_t>(m) * N + n;
        if (REF) {
            *c = alpha * v + beta * *c;
        } else {
            const float base = (beta == 0.0f) ? 0.0f : (beta == 1.0f) ? *c : *c * beta;
            *c = base + alpha * v;
        }
    }
}

template <bool REF, int MI, int NI, int KS>
void launch_tile(const float* A, const float* B, float* C, int batch, int M, int N, int K, float alpha, float beta,
                 hipStream_t s) {
    const int mt = ceil_div(M, 32 * MI), nt = ceil_div(N, 32 * NI);
    const dim3 grid(static_cast<unsigned>(mt) * static_cast<unsigned>(nt), 1, static_cast<unsigned>(batch));
    gemm_f32_kernel<REF, MI, NI, KS><<<grid, 64 * KS, 0, s>>>(A, B, C, M, N, K, mt, alpha, beta);
}

// Short K on many outputs: a 256-thread workgroup owns a 64x64 tile, each
// thread a 4x4 block of VALU sums, K staged 16 at a time.  The tiles above pay
// for eight partial tiles in LDS whatever K is.
// Where it wins, us (this / those; 8,937 shapes measured): K=16, M=512, N=2048
// 5.9 / 8.3, but M=64, N=257 5.3 / 3.4; K=48, M=512, N=2048 9.1 / 10.1; K=32,
// M=128, N=1024 6.8 / 3.1; K=80, M=2000, N=2048 19.9 / 22.8; M=2000, N=8192: K=96
// 64 / 75, K=192 111 / 115, K=256 142 / 130.  By valu_wins both together are
// 2.87 and 3.08 times as fast as this one alone over a grid of 2,184 shapes and
// 2,500 random ones, three of them more than 2.5% slower, by 5% at most (131 x 38
// x 192 x 16 (M, K, N, batch) 8.9 / 9.4).
// Its grid has two dimensions for the outputs, so it also takes those past
// 2^32 threads of the other's one.
constexpr int T = 64, TK = 16;

template <bool REF>
__global__ __launch_bounds__(256) void gemm_f32_valu_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                       float* __restrict__ C, int M, int N, int K, float alpha,
                                                       float beta) {
    __shared__ float sa[TK][T + 4];
    __shared__ float sb[TK][T + 4];
    const int64_t z = blockIdx.z;
    A += z * M * static_cast<int64_t>(K);
    B += z * K * static_cast<int64_t>(N);
    C += z * M * static_cast<int64_t>(N);
    const int m0 = blockIdx.y * T, n0 = blockIdx.x * T;
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    float acc[4][4] = {};
    for (int k0 = 0; k0 < K; k0 += TK) {
        for (int i = threadIdx.x; i < T * TK; i += 256) {
            const int r = i / TK, c = i % TK;  // A tile: 64 rows x 16 k
            const int gm = m0 + r, gk = k0 + c;
            sa[c][r] = (gm < M && gk < K) ? A[static_cast<int64_t>(gm) * K + gk] : 0.0f;
            const int kr = i / T, nc = i % T;  // B tile: 16 k x 64 cols
            const int gk2 = k0 + kr, gn = n0 + nc;
            sb[kr][nc] = (gk2 < K && gn < N) ? B[static_cast<int64_t>(gk2) * N + gn] : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < TK; ++kk) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = sa[kk][ty * 4 + i];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = sb[kk][tx * 4 + j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_fmaf(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int m = m0 + ty * 4 + i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + tx * 4 + j;
            if (n >= N) continue;
            float* c = C + static_cast<int64_t>(m) * N + n;
            if (REF) {
                *c = alpha * acc[i][j] + beta * *c;
            } else {
                const float base = (beta == 0.0f) ? 0.0f : (beta == 1.0f) ? *c : *c * beta;
                *c = base + alpha * acc[i][j];
            }
        }
    }
}

bool valu_wins(int batch, int M, int N, int K) {
    if (ceil_div(M, T) > 65535) return false;  // its grid's second dimension ends there
    if (static_cast<int64_t>(ceil_div(M, 64)) * ceil_div(N, 32) >= int64_t{1} << 24) return true;
    if (K < 24 && (M == 1 || N == 1)) return true;
    const int64_t tiles = static_cast<int64_t>(batch) * ceil_div(M, 32) * ceil_div(N, 32);
    const bool rows = M > 16;
    if (K < 32) return tiles > (rows && K >= 24 ? 512 : M < 3 ? 255 : 256);
    if (K < 64) return tiles > (!rows ? 256 : K == 32 ? 880 : 512);
    if (K < 96) return tiles > 1100;
    if (!rows && K % 32 != 0) return K < 256 && tiles > 2200;
    return K < 256 && tiles > (K < 128 && K % 32 != 0 ? 4000 : K < 200 ? 7900 : 14000);
}

template <bool REF>
int launch(const float* A, const float* B, float* C, int batch, int M, int N, int K, float alpha, float beta,
           void* stream, const char* who) {
    LHQ_REQUIRE(batch >= 0 && M >= 0 && N >= 0 && K >= 0, "%s: negative dims", who);
    LHQ_REQUIRE(batch <= 65535, "%s: batch %d too large", who, batch);
    if (batch == 0 || M == 0 || N == 0) return LHQ_OK;
    LHQ_REQUIRE(C && ((A && B) || K == 0), "%s: null pointer", who);
    hipStream_t s = as_stream(stream);
    static const int env = tuning_knob("LHQ_F32_VALU", -1);
    if (env < 0 ? valu_wins(batch, M, N, K) : env != 0) {
        gemm_f32_valu_kernel<REF><<<dim3(ceil_div(N, T), ceil_div(M, T), batch), 256, 0, s>>>(A, B, C, M, N, K, alpha,
                                                                                             beta);
        return check_launch(who);
    }
    auto tiles = [&](int rows, int cols) {
        return static_cast<int64_t>(batch) * ceil_div(M, rows) * ceil_div(N, cols);
    };
    // Measured (us, 64 x 32 tiles on 4 / 8 waves, 32 x 32 on 8; K = N = 4096):
    // M = 2048 712 / 726 / 818, M = 512 175 / 175 / 204, M = 100 55 / 51 / 58,
    // M = 64 50 / 47 / 30, M = 1 51 / 46 / 28: 64 rows per tile while every
    // CU still gets a workgroup, K over four waves once each gets four.
    if (tiles(64, 32) >= 1024) launch_tile<REF, 2, 1, 4>(A, B, C, batch, M, N, K, alpha, beta, s);
    else if (tiles(64, 32) >= 256) launch_tile<REF, 2, 1, 8>(A, B, C, batch, M, N, K, alpha, beta, s);
    else launch_tile<REF, 1, 1, 8>(A, B, C, batch, M, N, K, alpha, beta, s);
    return check_launch(who);
}

}  // namespace
}  // namespace lhq

extern "C" {

int lhq_gemm_f32(const float* A, const float* B, float* C, int M, int N, int K, float alpha, float beta,
                 void* stream) {
    return lhq::launch<false>(A, B, C, 1, M, N, K, alpha, beta, stream, "gemm_f32");
}

int lhq_gemm_f32_ref(const float* A, const float* B, float* C, int M, int N, int K, float alpha, float beta,
                     void* stream) {
    return lhq::launch<true>(A, B, C, 1, M, N, K, alpha, beta, stream, "gemm_f32_ref");
}

int lhq_gemm_f32_batched(const float* A, const float* B, float* C, int batch, int M, int N, int K, float alpha,
                         float beta, void* stream) {
    return lhq::launch<false>(A, B, C, batch, M, N, K, alpha, beta, stream, "gemm_f32_batched");
}

}  // extern "C"
