// FP64 LINPACK path: the reference built with DATA_TYPE=double (the "_DP"
// build, LINPACK/src/host/linpack_data.cpp:166-229 with HOST_DATA_TYPE
// double).  Same algorithm and storage as the FP32 path (row-major a,
// M = a^T, dgefa encoding without pivoting); the kernels:
//   * lu_f64_kernel: the 64 x 64 diagonal block in the registers of four waves
//     (lane c holds stored column c), pivots and multipliers broadcast with
//     v_readlane; the operation order of gefa_ref_nopvt with contraction off,
//     so the block is bit-identical to it;
//   * strip_f64_kernel: the top strip (two lanes per column of the strip,
//     the closed form of test_kernel_communication.cpp:776-789) and the left
//     strip (two lanes per row, :624-632) with the 64 values of the vector in
//     registers, coefficients from LDS; the left strip is also written
//     transposed (k-major) for the update;
//   * update_f64_kernel: C += Lt^T T on v_mfma_f64_16x16x4f64, 128 x 128
//     workgroup tiles of four 64 x 64 wave tiles, k-slabs of 16 through
//     double-buffered LDS, XCD-aware tile order as the FP32 update;
//   * gesl: one launch of a wave per 64 entries that pass solved blocks on, each
//     value its own flag; beyond what the device holds at once, per 64-block a one-wave
//     diagonal solve (block staged in LDS) and a column-parallel update of the
//     rest of x (the factor streamed once per sweep);
//   * residual r = b - M x with per-chunk partial sums added in fixed order.
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>
#include <cstdlib>

typedef double f64x4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int FB = 64;  // FP64 block size

__device__ __forceinline__ double bcast64(double v, int lane) {
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, lane);
    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), lane);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// ---------------------------------------------------------------- diagonal LU
// Stored row r of the block is M's column r; lane c of every wave belongs to
// column c, wave w holds the rows r with r % 4 = w.
//   for gk: D[gk][gk] = -1/D[gk][gk]; D[gk][c] *= D[gk][gk] (c > gk);
//           D[r][c] += D[gk][c] * D[r][gk] (r > gk, c > gk)
// Bound: the chain of 64 pivot steps -- a division, the scaled row through LDS
// to the other waves, one row's update.  The wave of the next pivot updates
// that row first, divides and publishes it, and catches up on its other rows
// behind the barrier, while the other waves are on theirs.  22 us; one wave
// holding all 64 rows took 36.
constexpr int LW = 4, LR = FB / LW;  // waves, rows per wave

__global__ __launch_bounds__(64 * LW) void lu_f64_kernel(double* __restrict__ A, int64_t lda,
                                                         int64_t off, int* __restrict__ status) {
#pragma clang fp contract(off)
    __shared__ double row[2][FB];
    const int c = threadIdx.x & 63, wave = threadIdx.x >> 6;
    double* base = A + off * lda + off;
    double d[LR];
#pragma unroll
    for (int i = 0; i < LR; ++i) d[i] = base[(int64_t)(LW * i + wave) * lda + c];
    bool bad = false;
    // row gk = LW i + (its wave), already updated by the steps before
    auto pivot = [&](double& x, int gk) {
        const double piv = bcast64(x, gk);
        const double inv = -1.0 / piv;
        bad |= (piv == 0.0) || !__builtin_isfinite(inv);
        x = (c > gk) ? x * inv : ((c == gk) ? inv : x);
        row[gk & 1][c] = x;
    };
    if (wave == 0) pivot(d[0], 0);
#pragma unroll
    for (int gk = 0; gk < FB; ++gk) {
        const int i0 = gk / LW, i1 = (gk + 1) / LW;
        __syncthreads();  // row gk is there; everyone is past row gk - 1
        if (gk + 1 == FB) break;
        const double u = row[gk & 1][c];
        if (wave == (gk + 1) % LW) {
            const double s = bcast64(d[i1], gk);
            if (c > gk) d[i1] = d[i1] + u * s;
            pivot(d[i1], gk + 1);
        } else if (wave > gk % LW) {
            // the wave's row LW i0 + wave > gk
            const double s = bcast64(d[i0], gk);
            if (c > gk) d[i0] = d[i0] + u * s;
        }
#pragma unroll
        for (int i = i0 + 1; i < LR; ++i) {
            if (i == i1 && wave == (gk + 1) % LW) continue;
            const double s = bcast64(d[i], gk);
            if (c > gk) d[i] = d[i] + u * s;
        }
    }
#pragma unroll
    for (int i = 0; i < LR; ++i) base[(int64_t)(LW * i + wave) * lda + c] = d[i];
    if (bad && c == 0 && status) atomicMax(status, 1);
}

// ---------------------------------------------------------------- strips
// 32 vectors per wave, each held by two lanes: half h of the wave has the
// elements e = 4 q + 2 h + b in x[2 q + b] (pairs, so that a row's elements
// move as 16-byte vectors).  Blocks [0, gtop) take top-strip columns, the rest
// left-strip rows, 128 vectors each.  The factored diagonal block lies in LDS
// in the order the lanes use it: S[k][h][2 q + b] = the coefficient of step k
// and element 4 q + 2 h + b, 16-byte broadcasts read one step ahead.
// Bound: the 64-step recurrence's instructions: 18 us, 46 with one vector per
// thread and 2016 scalar LDS reads each.  With both, GEFA at n = 8192 went
// from 17.2 to 13.5 ms (1024: 1.19 -> 0.72, 32768: 450 -> 437).
template <int H>
__device__ __forceinline__ double from_half64(double v) {
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint32_t l = (uint32_t)u, g = (uint32_t)(u >> 32);
    const auto a = __builtin_amdgcn_permlane32_swap(l, l, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(g, g, false, false);
    return __longlong_as_double((long long)(((uint64_t)b[H] << 32) | a[H]));
}

template <bool TOP>
__device__ __forceinline__ void strip_solve64(double (&x)[FB / 2], const double* S, int h) {
#pragma clang fp contract(off)
    const double* Sh = S + h * (FB / 2);
    double2 nx[2][FB / 4];
#pragma unroll
    for (int q = 0; q < FB / 4; ++q) nx[0][q] = *reinterpret_cast<const double2*>(Sh + 2 * q);
    // the scale of step k: element k's own coefficient
    auto dg_at = [&](int k) { return S[k * FB + ((k >> 1) & 1) * (FB / 2) + 2 * (k >> 2) + (k & 1)]; };
    double dg = TOP ? dg_at(0) : 0.0;
    static_for<0, FB>([&](auto kc) {
        constexpr int k = kc.value, q0 = k >> 2, kr = k & 3, hk = kr >> 1, ik = 2 * q0 + (k & 1);
        if constexpr (k + 1 < FB) {
#pragma unroll
            for (int q = (k + 1) >> 2; q < FB / 4; ++q)
                nx[(k + 1) & 1][q] = *reinterpret_cast<const double2*>(Sh + (k + 1) * FB + 2 * q);
        }
        double s = x[ik];
        if constexpr (TOP) s = s * dg;
        const double v = from_half64<hk>(s);
        if constexpr (TOP) {
            x[ik] = h == hk ? s : x[ik];
            if constexpr (k + 1 < FB) dg = dg_at(k + 1);
        }
        // the elements of k's own group of four that come after k
        if constexpr (kr < 2) {
            const double w = x[2 * q0] + v * nx[k & 1][q0].x;
            x[2 * q0] = h == 1 ? w : x[2 * q0];
        }
        if constexpr (kr < 3) {
            const double w = x[2 * q0 + 1] + v * nx[k & 1][q0].y;
            x[2 * q0 + 1] = kr == 0 || h == 1 ? w : x[2 * q0 + 1];
        }
#pragma unroll
        for (int q = q0 + 1; q < FB / 4; ++q) {
            const double2 f = nx[k & 1][q];
            x[2 * q] = x[2 * q] + v * f.x;
            x[2 * q + 1] = x[2 * q + 1] + v * f.y;
        }
        __builtin_amdgcn_sched_barrier(0);
    });
}

__global__ __launch_bounds__(256) void strip_f64_kernel(double* __restrict__ A, int64_t lda,
                                                        int64_t off, int64_t m, int gtop,
                                                        double* __restrict__ Lt, int64_t ldl) {
    __shared__ __attribute__((aligned(16))) double S[FB * FB];
    const int t = threadIdx.x;
    const double* D = A + off * lda + off;
    const bool top = (int)blockIdx.x < gtop;
    for (int e = t; e < FB * FB; e += 256) {
        const int i = e / FB, j = e % FB;
        // top: step j, element i; left: step i, element j
        const int k = top ? j : i, el = top ? i : j;
        S[k * FB + ((el >> 1) & 1) * (FB / 2) + 2 * (el >> 2) + (el & 1)] = D[(int64_t)i * lda + j];
    }
    __syncthreads();
    const int lane = t & 63, h = lane >> 5;
    const int64_t v = (int64_t)(top ? blockIdx.x : blockIdx.x - gtop) * 128 + (t >> 6) * 32 + (lane & 31);
    if (v >= m) return;  // m is a multiple of 64: whole waves
    double x[FB / 2];
    if (top) {
        // column off+FB+v of stored rows off..off+FB-1:
        //   for k: x_k *= D[k][k]; x_j += x_k * D[j][k] (j > k)
        double* col = A + (off + 2 * h) * lda + off + FB + v;
#pragma unroll
        for (int q = 0; q < FB / 4; ++q) {
            x[2 * q] = col[(int64_t)(4 * q) * lda];
            x[2 * q + 1] = col[(int64_t)(4 * q + 1) * lda];
        }
        strip_solve64<true>(x, S, h);
#pragma unroll
        for (int q = 0; q < FB / 4; ++q) {
            col[(int64_t)(4 * q) * lda] = x[2 * q];
            col[(int64_t)(4 * q + 1) * lda] = x[2 * q + 1];
        }
    } else {
        // stored row off+FB+v, columns off..off+FB-1:
        //   for k: x_i += x_k * D[k][i] (i > k)
        double* row = A + (off + FB + v) * lda + off + 2 * h;
#pragma unroll
        for (int q = 0; q < FB / 4; ++q) {
            const double2 p = *reinterpret_cast<const double2*>(row + 4 * q);
            x[2 * q] = p.x;
            x[2 * q + 1] = p.y;
        }
        strip_solve64<false>(x, S, h);
        double* lt = Lt + (int64_t)(2 * h) * ldl + v;
#pragma unroll
        for (int q = 0; q < FB / 4; ++q) {
            *reinterpret_cast<double2*>(row + 4 * q) = double2{x[2 * q], x[2 * q + 1]};
            lt[(int64_t)(4 * q) * ldl] = x[2 * q];
            lt[(int64_t)(4 * q + 1) * ldl] = x[2 * q + 1];
        }
    }
}

// ---------------------------------------------------------------- update
// C[r][c] += sum_k At[k][r] * Bt[k][c].  MFMA operand of lane l: A[l%16][l/16],
// B[l/16][l%16]; accumulator register q of lane l holds D[l/16 + 4q][l%16].
constexpr int UBM = 128, UBN = 128, UBK = 16, UNT = 512;
constexpr int UPAD = 16;  // LDS row = 144 doubles: the 4 k-rows of a read fall in distinct bank halves

__device__ __forceinline__ void tile_coords64(int bid, int nblk, int tiles_m, int tiles_n, int& tm,
                                              int& tn) {
    int pid = bid;
    if ((nblk & 7) == 0) pid = (bid & 7) * (nblk >> 3) + (bid >> 3);
    constexpr int GROUP = 8;
    const int per_group = GROUP * tiles_n;
    const int g = pid / per_group;
    const int first_m = g * GROUP;
    const int gsize = min(GROUP, tiles_m - first_m);
    const int in_g = pid - g * per_group;
    tm = first_m + in_g % gsize;
    tn = in_g / gsize;
}

// Slabs are staged with global_load_lds: each wave instruction moves one
// 1 KiB row of a slab (16 B per lane) to a wave-uniform LDS row; the padded
// LDS row keeps the four k-rows of an operand read in distinct bank halves.
// The accumulators start from C, so the epilogue is a plain store.  Eight
// waves of 64 x 32 per 128 x 128 tile, at most 128 VGPRs (four waves per
// SIMD, two workgroups per CU): 56.4-56.6 TFLOP/s at M = N = 16384-24576,
// K = 384, against 53.6-54.0 with four waves of 64 x 64 (two per SIMD); the
// DMA row pointers are formed once and advanced by a slab per step (1.9 of
// those 2.6 TFLOP/s).
__global__ __launch_bounds__(UNT, 4) void update_f64_kernel(double* __restrict__ C, int64_t ldc,
                                                            const double* __restrict__ At,
                                                            int64_t lda,
                                                            const double* __restrict__ Bt,
                                                            int64_t ldb, int M, int N, int K) {
    constexpr int FM = 4, FN = 2;  // 16 x 16 blocks per 64 x 32 wave tile
    constexpr int LDS_ROW = UBM + UPAD;
    constexpr int ROWS_PER_WAVE = UBK / (UNT / 64);  // slab rows each wave moves (2)
    __shared__ double As[2][UBK][LDS_ROW];
    __shared__ double Bs[2][UBK][LDS_ROW];
    const int tiles_m = (M + UBM - 1) / UBM, tiles_n = (N + UBN - 1) / UBN;
    int tm, tn;
    tile_coords64(blockIdx.x, tiles_m * tiles_n, tiles_m, tiles_n, tm, tn);
    const int m0 = tm * UBM, n0 = tn * UBN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave & 1, wn = wave >> 1;  // 2 x 4 waves
    const int l16 = lane & 15, lq = lane >> 4;
    const bool full = (m0 + UBM <= M) && (n0 + UBN <= N);
    // lane l moves doubles 2l, 2l+1 of a row; clamped so edge tiles read in
    // bounds (the clamped columns only reach rows/columns of C never stored)
    const int ca = min(2 * lane, M - m0 - 2), cb = min(2 * lane, N - n0 - 2);

    const double* pa0 = At + (int64_t)(wave * ROWS_PER_WAVE) * lda + m0 + ca;
    const double* pb0 = Bt + (int64_t)(wave * ROWS_PER_WAVE) * ldb + n0 + cb;
    auto dma_slab = [&](int k0, int buf) {
        const double* pa = pa0 + (int64_t)k0 * lda;
        const double* pb = pb0 + (int64_t)k0 * ldb;
#pragma unroll
        for (int s = 0; s < ROWS_PER_WAVE; ++s) {
            const int row = wave * ROWS_PER_WAVE + s;
            __builtin_amdgcn_global_load_lds(
                pa + s * lda, (__attribute__((address_space(3))) void*)(&As[buf][row][0]), 16, 0, 0);
            __builtin_amdgcn_global_load_lds(
                pb + s * ldb, (__attribute__((address_space(3))) void*)(&Bs[buf][row][0]), 16, 0, 0);
        }
    };
    const int rbase = m0 + wm * 64, cbase = n0 + wn * 32;
    f64x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int row = rbase + i * 16 + lq + 4 * q;
                const int col = cbase + j * 16 + l16;
                acc[i][j][q] = (full || (row < M && col < N)) ? C[(int64_t)row * ldc + col] : 0.0;
            }

    dma_slab(0, 0);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    const int nk = K / UBK;
    for (int kc = 0; kc < nk; ++kc) {
        const int buf = kc & 1;
        const bool more = kc + 1 < nk;
        if (more) dma_slab((kc + 1) * UBK, buf ^ 1);
#pragma unroll
        for (int kq = 0; kq < UBK / 4; ++kq) {
            double a[FM], b[FN];
#pragma unroll
            for (int i = 0; i < FM; ++i) a[i] = As[buf][kq * 4 + lq][wm * 64 + i * 16 + l16];
#pragma unroll
            for (int j = 0; j < FN; ++j) b[j] = Bs[buf][kq * 4 + lq][wn * 32 + j * 16 + l16];
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        if (more) {
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
        }
    }
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int row = rbase + i * 16 + lq + 4 * q;
                const int col = cbase + j * 16 + l16;
                if (full || (row < M && col < N)) C[(int64_t)row * ldc + col] = acc[i][j][q];
            }
}

// The update of small regions, as the FP32 one (gemm.hip): a wave owns a 16 x
// 32 block of C and reads its operands straight into the MFMA registers, 16 k
// values at a time, three chunks ahead; four waves (32 x 64 of C) share them
// through the CU's L1.  The row and column blocks on a step's critical path
// are 64 wide: the tiled kernel, one 128 x 128 tile per CU and half of it
// empty, takes 68 us for K = 640, all of it one CU's matrix rate.
// Bound: one memory round trip, then the wave's chain of K / 2 MFMAs (64
// cycles each).  C first, then k in order: the bits of the tiled kernel.
struct Region64 {
    double* C;
    const double* At;
    const double* Bt;
    int M, N;
};
constexpr int SCH = 4;   // 16 k values: 4 MFMA steps per chunk
constexpr int SBUF = 4;

__global__ __launch_bounds__(256) void update_small_f64_kernel(Region64 g, int64_t ldc, int64_t lda,
                                                               int64_t ldb, int K, Region64 g2) {
    int tiles_n = (g.N + 63) / 64, bid = blockIdx.x;
    const int nblk = ((g.M + 31) / 32) * tiles_n;
    if (bid >= nblk) {  // second region
        bid -= nblk;
        g = g2;
        tiles_n = (g.N + 63) / 64;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = lane & 15, kk = lane >> 4;
    const int m0 = (bid / tiles_n) * 32 + (wave & 1) * 16;
    const int n0 = (bid % tiles_n) * 64 + (wave >> 1) * 32;
    if (m0 >= g.M || n0 >= g.N) return;  // regions are whole 16 x 32 blocks
    const double* a = g.At + (int64_t)kk * lda + m0 + c;
    const double* b = g.Bt + (int64_t)kk * ldb + n0 + c;
    double va[SBUF][SCH], vb[SBUF][SCH][2];
    auto load = [&](int ch, int buf) {
#pragma unroll
        for (int i = 0; i < SCH; ++i) {
            const int64_t k = 4 * (ch * SCH + i);
            va[buf][i] = a[k * lda];
            vb[buf][i][0] = b[k * ldb];
            vb[buf][i][1] = b[k * ldb + 16];
        }
    };
    // accumulator register q: row kk + 4 q
    double* p = g.C + (int64_t)(m0 + kk) * ldc + n0 + c;
    f64x4 acc[2];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        acc[0][q] = p[(int64_t)(4 * q) * ldc];
        acc[1][q] = p[(int64_t)(4 * q) * ldc + 16];
    }
    const int nch = K / (4 * SCH);
#pragma unroll
    for (int u = 0; u < SBUF - 1; ++u)
        if (u < nch) load(u, u);
    for (int ch0 = 0; ch0 < nch; ch0 += SBUF) {
#pragma unroll
        for (int u = 0; u < SBUF; ++u) {
            const int ch = ch0 + u;
            if (ch >= nch) break;
            if (ch + SBUF - 1 < nch) load(ch + SBUF - 1, (u + SBUF - 1) % SBUF);
#pragma unroll
            for (int i = 0; i < SCH; ++i) {
                acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(va[u][i], vb[u][i][0], acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(va[u][i], vb[u][i][1], acc[1], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        p[(int64_t)(4 * q) * ldc] = acc[0][q];
        p[(int64_t)(4 * q) * ldc + 16] = acc[1][q];
    }
}

// ---------------------------------------------------------------- substitution
// forward, block q (64 entries from k0): x_i += x_k * a[k][i] (k < i, inside
// the block), the block staged in LDS, one wave; then x_i += sum_{k in block}

// The 64 x 64 diagonal block at (k0, k0) into S, one column per lane, with
// all 64 loads of a lane in flight before the first is stored.
__device__ __forceinline__ void load_block64(const double* __restrict__ A, int64_t lda, int64_t k0,
                                             double (*S)[FB + 1]) {
    const int l = threadIdx.x;
    double v[FB];
#pragma unroll
    for (int r = 0; r < FB; ++r) v[r] = A[(k0 + r) * lda + k0 + l];
#pragma unroll
    for (int r = 0; r < FB; ++r) S[r][l] = v[r];
    __syncthreads();
}

// x_k * a[k][i] for i >= k0 + 64.
__global__ __launch_bounds__(64) void gesl_diag_fwd_f64(const double* __restrict__ A, int64_t lda,
                                                        int64_t k0, double* __restrict__ x) {
#pragma clang fp contract(off)
    __shared__ double S[FB][FB + 1];
    const int l = threadIdx.x;
    load_block64(A, lda, k0, S);
    double xi = x[k0 + l];
    for (int k = 0; k < FB - 1; ++k) {
        const double xk = bcast64(xi, k);
        if (l > k) xi = xi + xk * S[k][l];
    }
    x[k0 + l] = xi;
}

// backward, block at k0: for k = k0+63 .. k0: s = x_k * a[k][k]; x_k = -s;
// x_i += s * a[k][i] (k0 <= i < k)
__global__ __launch_bounds__(64) void gesl_diag_bwd_f64(const double* __restrict__ A, int64_t lda,
                                                        int64_t k0, double* __restrict__ x) {
#pragma clang fp contract(off)
    __shared__ double S[FB][FB + 1];
    const int l = threadIdx.x;
    load_block64(A, lda, k0, S);
    double xi = x[k0 + l];
    for (int k = FB - 1; k >= 0; --k) {
        const double s = bcast64(xi, k) * S[k][k];
        if (l == k) xi = -s;
        if (l < k) xi = xi + s * S[k][l];
    }
    x[k0 + l] = xi;
}

// x_i += sum over the block's k of s_k * a[k][i] for i in [i0, i1), in
// gesl_ref_nopvt's order: forward s_k = x_k, k increasing; backward the block
// holds x_k = -s_k, so s_k = -x_k, k decreasing.
template <bool BWD>
__global__ __launch_bounds__(256) void gesl_gemv_f64(const double* __restrict__ A, int64_t lda,
                                                     int64_t k0, int64_t i0, int64_t i1,
                                                     double* __restrict__ x) {
#pragma clang fp contract(off)
    __shared__ double xs[FB];
    if (threadIdx.x < FB) xs[threadIdx.x] = BWD ? -x[k0 + threadIdx.x] : x[k0 + threadIdx.x];
    __syncthreads();
    const int64_t i = i0 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= i1) return;
    // the block's 64 factor entries of column i, all in flight at once
    double a[FB];
#pragma unroll
    for (int u = 0; u < FB; ++u) a[u] = A[(k0 + (BWD ? FB - 1 - u : u)) * lda + i];
    double acc = x[i];
#pragma unroll
    for (int u = 0; u < FB; ++u) {
        const int k = BWD ? FB - 1 - u : u;
        acc = acc + xs[k] * a[u];
    }
    x[i] = acc;
}

// Single-launch substitution: one wave per 64 entries, which stay in its
// registers (lane l, entry l).  Forward, it takes block q's contribution as
// soon as q is solved, q ascending, then solves its own block; backward the
// same descending.  The arithmetic and its order are those of the kernels
// above.  A solved block is published by agent-scope stores; an entry not yet
// there holds kEmpty64, a NaN pattern that no published value has (a small
// kernel fills it in before), so the values are their own flags.  Waits are
// bounded and a wave that gives up raises status bit 2 and leaves; the host
// then solves launch after launch.  The tile of a contribution (and the wave's
// own diagonal block, the same access) is loaded into the registers that the
// tile before it leaves, so only the arithmetic follows a wait.
// Bound: the chain of 2 n / 64 block solves, each a value's trip, 64 steps of
// contribution and 64 of the solve.  0.91 ms at n = 8192, 2.92 launch after
// launch, 4 n / 64 of them (n = 1024 0.31 -> 0.11, 32768 12.5 -> 4.3); with
// drained stores, flags and then the values 1.00, 0.124 and 4.7.
// Polls before a wave gives up, about a second: whoever waits that long shares
// the device with launches that keep its partners from starting, and solving
// launch after launch takes milliseconds.
constexpr long kGesl64SpinLimit = 1L << 20;

constexpr unsigned long long kEmpty64 = ~0ull;

__global__ void gesl_reset_f64(double* __restrict__ w, int64_t count, int* __restrict__ status) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < count) w[i] = __longlong_as_double((long long)kEmpty64);
    if (i == 0) *status = 0;
}

__global__ __launch_bounds__(64) void gesl_persist_f64(const double* __restrict__ A, int64_t lda,
                                                       int N, double* __restrict__ x,
                                                       double* __restrict__ pf,
                                                       double* __restrict__ pb,
                                                       int* __restrict__ status, long spin_limit) {
#pragma clang fp contract(off)
    const int l = threadIdx.x, s = blockIdx.x;
    const double* col = A + (int64_t)s * FB + l;  // this lane's column of the factor
    auto put = [&](double* p, double v) {
        const unsigned long long u = (unsigned long long)__double_as_longlong(v);
        __hip_atomic_store(reinterpret_cast<unsigned long long*>(p + (int64_t)s * FB + l),
                           u == kEmpty64 ? 0x7ff8000000000000ull : u, __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    };
    // this lane's entry of block q once all of them are there; true: gave up
    auto get = [&](const double* p, int q, double& v) {
        for (long spins = 1;; ++spins) {
            const unsigned long long u = __hip_atomic_load(
                reinterpret_cast<const unsigned long long*>(p + (int64_t)q * FB + l),
                __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            v = __longlong_as_double((long long)u);
            if (!__any(u == kEmpty64)) return false;
            if (spins > spin_limit ||
                ((spins & 31) == 0 &&
                 (__hip_atomic_load(status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & 2))) {
                if (l == 0) atomicOr(status, 2);
                return true;
            }
            // on the chain only the next block's wave waits
            if (q + 1 != s && q - 1 != s) __builtin_amdgcn_s_sleep(1);
        }
    };
    double a[FB];
    auto load = [&](int q) {
#pragma unroll
        for (int u = 0; u < FB; ++u) a[u] = col[((int64_t)q * FB + u) * lda];
    };
    double xi = x[(int64_t)s * FB + l];
    // ---- forward: L y = b
    load(0);
    for (int q = 0; q < s; ++q) {
        double xs;
        if (get(pf, q, xs)) return;
        const double* next = col + (int64_t)(q + 1) * FB * lda;
#pragma unroll
        for (int u = 0; u < FB; ++u) {
            xi = xi + bcast64(xs, u) * a[u];
            a[u] = next[u * lda];
        }
    }
#pragma unroll
    for (int k = 0; k < FB - 1; ++k) {
        const double xk = bcast64(xi, k);
        if (l > k) xi = xi + xk * a[k];
    }
    put(pf, xi);
    // ---- backward: U x = y
    load(N - 1);
    for (int q = N - 1; q > s; --q) {
        double xs;
        if (get(pb, q, xs)) return;
        xs = -xs;
        const double* next = col + (int64_t)(q - 1) * FB * lda;
#pragma unroll
        for (int u = FB - 1; u >= 0; --u) {
            xi = xi + bcast64(xs, u) * a[u];
            a[u] = next[u * lda];
        }
    }
#pragma unroll
    for (int k = FB - 1; k >= 0; --k) {
        const double sk = bcast64(xi, k) * bcast64(a[k], k);
        if (l == k) xi = -sk;
        if (l < k) xi = xi + sk * a[k];
    }
    put(pb, xi);
    x[(int64_t)s * FB + l] = xi;
}

// ---------------------------------------------------------------- residual
// partial[c][i] = sum_{j in chunk c} M(i, j) x_j, M(i, j) = A[j][i]
constexpr int RCH64 = 256;
__global__ void resid_partial_f64(const double* __restrict__ A, int64_t lda, int64_t n,
                                  const double* __restrict__ x, double* __restrict__ part) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t c = blockIdx.y;
    if (i >= n) return;
    const int64_t j0 = c * RCH64, j1 = min(n, j0 + RCH64);
    double s = 0.0, a = 0.0;
    for (int64_t j = j0; j < j1; ++j) {
        const double v = A[j * lda + i];
        s = fma(v, x[j], s);
        a += fabs(v);
    }
    part[(2 * c) * n + i] = s;
    part[(2 * c + 1) * n + i] = a;
}

// out = (||b - Mx||inf, ||M||inf, ||x||inf, ||b||inf), one workgroup
__global__ __launch_bounds__(256) void resid_final_f64(const double* __restrict__ part,
                                                       int64_t nch, int64_t n,
                                                       const double* __restrict__ x,
                                                       const double* __restrict__ b,
                                                       double* __restrict__ out) {
    __shared__ double red[4][256];
    double m[4] = {0, 0, 0, 0};
    for (int64_t i = threadIdx.x; i < n; i += 256) {
        double s = 0.0, a = 0.0;
        for (int64_t c = 0; c < nch; ++c) {
            s += part[(2 * c) * n + i];
            a += part[(2 * c + 1) * n + i];
        }
        m[0] = fmax(m[0], fabs(b[i] - s));
        m[1] = fmax(m[1], a);
        m[2] = fmax(m[2], fabs(x[i]));
        m[3] = fmax(m[3], fabs(b[i]));
    }
    for (int q = 0; q < 4; ++q) red[q][threadIdx.x] = m[q];
    __syncthreads();
    if (threadIdx.x < 4) {
        double v = 0.0;
        for (int u = 0; u < 256; ++u) v = fmax(v, red[threadIdx.x][u]);
        out[threadIdx.x] = v;
    }
}

__global__ void f32_to_f64_kernel(const float* __restrict__ s, int64_t lds, double* __restrict__ d,
                                  int64_t ldd, int64_t n) {
    for (int64_t r = blockIdx.y; r < n; r += gridDim.y)
        for (int64_t c = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; c < n;
             c += (int64_t)gridDim.x * blockDim.x)
            d[r * ldd + c] = (double)s[r * lds + c];
}

}  // namespace

int f64_block() { return FB; }

hipError_t launch_lu_f64(double* A, int64_t lda, int64_t off, int* status, hipStream_t s) {
    lu_f64_kernel<<<1, 64 * LW, 0, s>>>(A, lda, off, status);
    return hipGetLastError();
}

hipError_t launch_strips_f64(double* A, int64_t lda, int64_t off, int64_t m, double* Lt,
                             int64_t ldl, hipStream_t s) {
    if (m <= 0) return hipSuccess;
    if (m % 32) return hipErrorInvalidValue;
    const int g = (int)((m + 127) / 128);
    strip_f64_kernel<<<2 * g, 256, 0, s>>>(A, lda, off, m, g, Lt, ldl);
    return hipGetLastError();
}

hipError_t launch_update_f64(double* C, int64_t ldc, const double* Lt, int64_t ldl,
                             const double* T, int64_t ldt, int M, int N, double* C2,
                             const double* Lt2, const double* T2, int M2, int N2, int K,
                             hipStream_t s) {
    if (M <= 0 || N <= 0) M = N = 0;
    if (M2 <= 0 || N2 <= 0) M2 = N2 = 0;
    if (!M && !M2) return hipSuccess;
    if (K % UBK || (M & 1) || (N & 1) || (M2 & 1) || (N2 & 1)) return hipErrorInvalidValue;
    const auto tiles = [](int m, int n, int tm, int tn) {
        return ((m + tm - 1) / tm) * ((n + tn - 1) / tn);
    };
    const int t1 = tiles(M, N, UBM, UBN), t2 = tiles(M2, N2, UBM, UBN);
    // One or two 64-wide blocks (half a tile each) up to two tiles per CU, other
    // regions while half the CUs would have no tile: with every region up to
    // 128 tiles on the small path GEFA at n = 8192 takes 17.2 ms, up to 256
    // 17.8, up to 512 18.7 (none: 33.5); n = 16384 89.5, 73.5, 74.0 (99.3) and
    // n = 32768 464.6, 459.1, 449.7 (474.2), where the row and column blocks
    // make up the larger counts.
    const bool narrow = std::min(M, N) <= FB && std::min(M2, N2) <= FB;
    if (t1 + t2 <= (narrow ? 512 : 128) && M % 16 == 0 && N % 32 == 0 && M2 % 16 == 0 && N2 % 32 == 0) {
        update_small_f64_kernel<<<(unsigned)(tiles(M, N, 32, 64) + tiles(M2, N2, 32, 64)), 256, 0,
                                  s>>>(Region64{C, Lt, T, M, N}, ldc, ldl, ldt, K,
                                       Region64{C2, Lt2, T2, M2, N2});
        return hipGetLastError();
    }
    if (t1) update_f64_kernel<<<t1, UNT, 0, s>>>(C, ldc, Lt, ldl, T, ldt, M, N, K);
    if (t2) update_f64_kernel<<<t2, UNT, 0, s>>>(C2, ldc, Lt2, ldl, T2, ldt, M2, N2, K);
    return hipGetLastError();
}

int64_t gesl_f64_work(int64_t n) {
    // both sweeps' published blocks, the status
    return 2 * n + 8;
}

const int* gesl_f64_status(const double* work, int64_t n) {
    return reinterpret_cast<const int*>(work + 2 * n);
}

hipError_t launch_gesl_f64(const double* A, int64_t lda, int64_t n, double* x, double* work,
                           hipStream_t s, bool per_block) {
    if (n % FB) return hipErrorInvalidValue;
    int* status = reinterpret_cast<int*>(work + 2 * n);
    const int64_t N = n / FB;
    // Every wave has to be resident at once: at most half of what the device
    // holds, so that other work on it leaves room (n up to 65536), and at most
    // HPL_GESL_GROUPS; beyond, where the device does not say, or where the
    // caller asks for it (per_block), launch after launch.
    if (!per_block) {
        int per_cu = 0, dev = 0, cus = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                &per_cu, reinterpret_cast<const void*>(gesl_persist_f64), 64, 0) != hipSuccess ||
            hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) !=
                hipSuccess) {
            (void)hipGetLastError();
            per_cu = cus = 0;
        }
        gesl_reset_f64<<<(unsigned)((2 * n + 255) / 256), 256, 0, s>>>(work, 2 * n, status);
        int64_t most = (int64_t)per_cu * cus / 2;
        if (const char* e = getenv("HPL_GESL_GROUPS")) most = std::min<int64_t>(most, atoll(e));
        if (N <= most) {
            gesl_persist_f64<<<(unsigned)N, 64, 0, s>>>(A, lda, (int)N, x, work, work + n, status,
                                                        gesl_spin_limit(kGesl64SpinLimit));
            return hipGetLastError();
        }
    }
    for (int64_t k0 = 0; k0 < n; k0 += FB) {
        gesl_diag_fwd_f64<<<1, 64, 0, s>>>(A, lda, k0, x);
        const int64_t i0 = k0 + FB;
        if (i0 < n)
            gesl_gemv_f64<false><<<(unsigned)((n - i0 + 255) / 256), 256, 0, s>>>(A, lda, k0, i0,
                                                                                  n, x);
    }
    for (int64_t k0 = n - FB; k0 >= 0; k0 -= FB) {
        gesl_diag_bwd_f64<<<1, 64, 0, s>>>(A, lda, k0, x);
        if (k0 > 0)
            gesl_gemv_f64<true><<<(unsigned)((k0 + 255) / 256), 256, 0, s>>>(A, lda, k0, 0, k0, x);
    }
    return hipGetLastError();
}

int64_t residual_f64_work(int64_t n) { return 2 * ((n + RCH64 - 1) / RCH64) * n; }

hipError_t launch_residual_f64(const double* A, int64_t lda, int64_t n, const double* x,
                               const double* b, double* work, double* out4, hipStream_t s) {
    const int64_t nch = (n + RCH64 - 1) / RCH64;
    resid_partial_f64<<<dim3((unsigned)((n + 255) / 256), (unsigned)nch), 256, 0, s>>>(A, lda, n, x,
                                                                                    work);
    resid_final_f64<<<1, 256, 0, s>>>(work, nch, n, x, b, out4);
    return hipGetLastError();
}

hipError_t launch_f32_to_f64(const float* src, int64_t lds, double* dst, int64_t ldd, int64_t n,
                             hipStream_t s) {
    dim3 g((unsigned)std::min<int64_t>((n + 255) / 256, 64), (unsigned)std::min<int64_t>(n, 8192));
    f32_to_f64_kernel<<<g, 256, 0, s>>>(src, lds, dst, ldd, n);
    return hipGetLastError();
}
