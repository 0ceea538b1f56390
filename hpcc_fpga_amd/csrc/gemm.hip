// Trailing-matrix update ("inner_update_mm", LINPACK/src/device/hpl_torus_PCIE.cl:711-865).
//
// C[r][c] += sum_k Lt[k][r] * T[k][c]   for r < M, c < N, k < K
// C is the row-major trailing matrix (ldc), Lt the transposed left strips
// written by the panel solves (k-major, ldl) and T the top strips as they lie
// in A (k-major, ldt).  With the multipliers stored negated this is exactly
// the reference's C += Left * Top (alpha = beta = +1).  K is a multiple of the
// block size: the schedule may apply several steps' updates in one launch.
//
// Tile 128 x 128 with 16-deep k slabs and eight wave64s of 32 x 64 (two
// v_mfma_f32_32x32x2_f32 blocks each), 32 KiB of LDS per workgroup, four
// waves per SIMD, slabs staged by LDS DMA.  Measured on MI355X against nine
// other tile shapes at M = N = 16384 and 32256, K = 256 and 512: 111-113
// TFLOP/s at K = 256 and 121 at K = 512 with register staging (the 32-deep
// version of the same tile: 88-103 and 103-119); DMA staging adds 2-4%
// (114.5-115.6 and 121.6-125.4) with bit-identical results.
#include "gemm_kernel.hpp"
#include "kernels.hpp"

namespace {

// The update of small regions: a wave owns a 32 x 32 block of C and reads its
// operands straight into the registers of v_mfma_f32_32x32x2_f32 (lane l: k
// row l / 32, column l % 32: two 128-byte row segments per load), 16 k values
// at a time, three chunks ahead; no LDS, no barrier.  Four waves (64 x 64 of
// C) share the segments through the CU's L1.
// The tiled kernel above takes 20 us for one 128 x 128 tile at K = 128 -- a
// memory round trip per 16-deep slab, then 6.8 us of one CU's matrix rate --
// and a step's critical path holds such launches of one to a few dozen tiles.
// Bound: one memory round trip, then the wave's chain of K / 2 MFMAs (64
// cycles each).  C first, then the k pairs in order: the bits of the tiled
// kernel.
constexpr int kChunk = 8;  // k pairs per chunk
constexpr int kBufs = 4;

__global__ __launch_bounds__(256) void update_small_kernel(
    float* __restrict__ C, int64_t ldc, const float* __restrict__ At, int64_t lda,
    const float* __restrict__ Bt, int64_t ldb, int M, int N, int K, gemm_f32::Region r2) {
    int tiles_n = (N + 63) / 64, bid = blockIdx.x;
    const int nblk = ((M + 63) / 64) * tiles_n;
    if (bid >= nblk) {  // second region
        bid -= nblk;
        C = r2.C;
        At = r2.At;
        Bt = r2.Bt;
        M = r2.M;
        N = r2.N;
        tiles_n = (N + 63) / 64;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int lr = lane & 31, lh = lane >> 5;
    const int m0 = (bid / tiles_n) * 64 + (wave & 1) * 32;
    const int n0 = (bid % tiles_n) * 64 + (wave >> 1) * 32;
    if (m0 >= M || n0 >= N) return;  // regions are whole 32 x 32 blocks

    const float* a = At + (int64_t)lh * lda + m0 + lr;
    const float* b = Bt + (int64_t)lh * ldb + n0 + lr;
    float va[kBufs][kChunk], vb[kBufs][kChunk];
    auto load = [&](int ch, int buf) {
#pragma unroll
        for (int i = 0; i < kChunk; ++i) {
            va[buf][i] = a[(int64_t)(2 * (ch * kChunk + i)) * lda];
            vb[buf][i] = b[(int64_t)(2 * (ch * kChunk + i)) * ldb];
        }
    };
    float* c = C + (int64_t)m0 * ldc + n0 + lr;
    f32x16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = c[(int64_t)acc_row(r, lane) * ldc];
    const int nch = K / (2 * kChunk);
#pragma unroll
    for (int p = 0; p < kBufs - 1; ++p)
        if (p < nch) load(p, p);
    for (int ch0 = 0; ch0 < nch; ch0 += kBufs) {
#pragma unroll
        for (int p = 0; p < kBufs; ++p) {
            const int ch = ch0 + p;
            if (ch >= nch) break;
            if (ch + kBufs - 1 < nch) load(ch + kBufs - 1, (p + kBufs - 1) % kBufs);
#pragma unroll
            for (int i = 0; i < kChunk; ++i) acc = mfma32(va[p][i], vb[p][i], acc);
        }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) c[(int64_t)acc_row(r, lane) * ldc] = acc[r];
}

}  // namespace

hipError_t launch_gemm_update_f32_2(float* C, int64_t ldc, const float* Lt, int64_t ldl,
                                    const float* T, int64_t ldt, int M, int N, float* C2,
                                    const float* Lt2, const float* T2, int M2, int N2, int K,
                                    hipStream_t s) {
    const gemm_f32::Region r2{C2, Lt2, T2, M2 > 0 && N2 > 0 ? M2 : 0, M2 > 0 && N2 > 0 ? N2 : 0};
    const auto tiles = [](int64_t m, int64_t n, int64_t t) {
        return ((m + t - 1) / t) * ((n + t - 1) / t);
    };
    // Up to one 128 x 128 tile per CU the tiled kernel leaves the chip idle (a
    // CU holds two of its workgroups); past that its operand reuse wins: n =
    // 7488, block 64: 10.94 ms without this path, 9.97 up to 4 tiles, 9.90 up
    // to 64, 9.73 up to 256, 10.32 up to 600; n = 32768: 202.3, 201.7, 202.1,
    // 201.4, 206.6; n = 2048: 2.01, 1.86, 1.68, 1.70, 1.68.
    constexpr int64_t kMaxTiles = 256;
    if (M > 0 && N > 0 && M % 32 == 0 && N % 32 == 0 && r2.M % 32 == 0 && r2.N % 32 == 0 &&
        K % (2 * kChunk) == 0 && tiles(M, N, 128) + tiles(r2.M, r2.N, 128) <= kMaxTiles) {
        const unsigned grid = (unsigned)(tiles(M, N, 64) + tiles(r2.M, r2.N, 64));
        update_small_kernel<<<grid, 256, 0, s>>>(C, ldc, Lt, ldl, T, ldt, M, N, K, r2);
        return hipGetLastError();
    }
    return gemm_f32::launch2<128, 128, 16, 32, 64, 2, false, false, true>(C, ldc, Lt, ldl, T, ldt,
                                                                          M, N, K, r2, s);
}

hipError_t launch_gemm_update_f32(float* C, int64_t ldc, const float* Lt, int64_t ldl,
                                  const float* T, int64_t ldt, int M, int N, int K,
                                  hipStream_t s) {
    return launch_gemm_update_f32_2(C, ldc, Lt, ldl, T, ldt, M, N, nullptr, nullptr, nullptr, 0, 0,
                                    K, s);
}
