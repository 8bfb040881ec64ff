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
// walked all of K took 550); M = 1 28 us, 2.4 TB/s of B (502); M = 512 175 us,
// 98 TFLOP/s (584).
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
    // column strip go to one XCD, whose L2 then reads the strip's B once
    const int xcd = blockIdx.x % kXcds, id = blockIdx.x / kXcds;
    const int m0 = (id % mt) * 32 * MI;
    const int n0 = ((id / mt) * kXcds + xcd) * 32 * NI;
    if (n0 >= N) return;  // uniform per workgroup
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
            for (int q = 0; q < 4; ++q) r.a[i][q] = load_f32x4<full.value>(ap[i][q] + k0, K - k0 - 4 * ac);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const int k = k0 + 8 * t, left = K - k - 4 * h;  // the lane's live k from here on
#pragma unroll
            for (int j = 0; j < NI; ++j)
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    r.b[j][t][u] = full.value || u < left ? bp[j][static_cast<int64_t>(k + u) * N] : 0.0f;
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
        f32x4_t a[MI][4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int i = 0; i < MI; ++i)
                a[i][t] = *reinterpret_cast<const f32x4_t*>(mine + (32 * i + l) * kStage + 4 * ((2 * t + h) ^ (l & 7)));
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
    const dim3 grid(static_cast<unsigned>(static_cast<int64_t>(mt) * ceil_div(nt, kXcds) * kXcds), 1,
                    static_cast<unsigned>(batch));
    gemm_f32_kernel<REF, MI, NI, KS><<<grid, 64 * KS, 0, s>>>(A, B, C, M, N, K, mt, alpha, beta);
}

template <bool REF>
int launch(const float* A, const float* B, float* C, int batch, int M, int N, int K, float alpha, float beta,
           void* stream, const char* who) {
    LHQ_REQUIRE(batch >= 0 && M >= 0 && N >= 0 && K >= 0, "%s: negative dims", who);
    LHQ_REQUIRE(batch <= 65535, "%s: batch %d too large", who, batch);
    if (batch == 0 || M == 0 || N == 0) return LHQ_OK;
    LHQ_REQUIRE(C && ((A && B) || K == 0), "%s: null pointer", who);
    hipStream_t s = as_stream(stream);
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
