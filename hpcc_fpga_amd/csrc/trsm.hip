// Panel triangular solves: "top_update" and "left_update"
// (LINPACK/src/device/hpl_torus_PCIE.cl:452-582 and :588-709).
//
// After the diagonal block D (row-major, B x B) of step k is factorised, the
// row-major strip right of it ("top" blocks, M's L-panel) and the strip below
// it ("left" blocks, M's U-panel) are solved.  Both are a forward substitution
// applied to many independent vectors v of length B:
//     y_i = (v_i + sum_{p<i} C[i][p] y_p) * s_i,   i = 0..B-1
//   top : vectors = columns of the strip, C[i][p] = D[i][p], s_i = D[i][i]
//         (closed form of LINPACK/tests/test_kernel_communication.cpp:776-789)
//   left: vectors = rows of the strip,    C[i][p] = D[p][i], s_i = 1
//         (closed form of test_kernel_communication.cpp:624-632)
// The left strip is also written transposed (k-major) for the trailing GEMM,
// as the reference's left_update writes its transposed copy
// (hpl_torus_PCIE.cl:697-708).
//
// Mixed precision: the solved strips can also be written as BF16/FP16 copies
// (k-contiguous) or as FP8 E4M3 copies with one power-of-two scale per block
// of 32 vectors x B (the block's amax maps to at most 448, so the scaling is
// exact and nothing saturates).
//
// Blocking: rows are taken 32 at a time.  For block q the contribution of the
// already solved rows is a 32 x 32q by 32q x 32 product on MFMA
// (v_mfma_f32_32x32x2_f32), and the 32 x 32 diagonal system is applied as its
// precomputed inverse G_q = (S^-1 - C_qq)^-1, also on MFMA.  Either one
// wavefront owns 32 vectors for all B rows, so that no workgroup barrier is
// needed, or (trsm_split_kernel) several share them.
#include "common.hpp"
#include "kernels.hpp"

#include <type_traits>

namespace {

// ----------------------------------------------------------------------------
// prep: transposed copy of D (coefficients of the top solve become coalesced)
// and the 32 x 32 inverses of the diagonal sub-systems, stored transposed:
//   inv + 0*NQ*1024 : G^T for top   (S^-1 - C)^-1 with C = D lower, s = diag D
//   inv + 1*NQ*1024 : G^T for left  (I - C)^-1 with C[i][p] = D[p][i]
//   inv + 2*NQ*1024 : H^T for the back substitution of GESL, H = U_qq^-1 with
//                     U[i][p] = D[p][i] (p > i), 1/u_ii = -D[i][i]: the
//                     negated transpose of the first
// Launch: two waves per inverse of the first two types, then one workgroup per
// 32 x 32 block of the copy (with DT); grid.y the diagonal blocks.
//
// Bound: the recurrence of the unit vectors, x_r += x_j S[j][r] for r > j, 32
// steps of one wave.  An element per lane of a DPP row: lane (r, g) of wave w
// holds elements r and 16 + r of vectors 16 w + 4 g + k, a step is a broadcast
// and a masked FMA per register, and the first half's part of the second is
// taken over the solved elements at once; wave 1's vectors have no first half.
// (A column of the inverse per lane, all three types: 8.2 us at n = 1024, 5.2
// here; hpl_gesl_noalloc there 47.3 -> 42.6 us with the clearing here.)
//
// pf, pb, status: the substitution's shares, cleared for a launch that follows.
// ----------------------------------------------------------------------------
// d[k] += m[k] s in the lanes that the mask M has in each half of the wave (every
// lane of the wave is active here; early clobbers and s_nop as in lu.hip's add_in)
template <unsigned M>
__device__ __forceinline__ void fma_in(float (&d)[4], const float (&m)[4], float s) {
    asm("s_mov_b32 exec_lo, %9\n\ts_mov_b32 exec_hi, %9\n\t"
        "v_fmac_f32 %0, %4, %8\n\tv_fmac_f32 %1, %5, %8\n\t"
        "v_fmac_f32 %2, %6, %8\n\tv_fmac_f32 %3, %7, %8\n\ts_mov_b64 exec, -1\n\ts_nop 0"
        : "+&v"(d[0]), "+&v"(d[1]), "+&v"(d[2]), "+&v"(d[3])
        : "v"(m[0]), "v"(m[1]), "v"(m[2]), "v"(m[3]), "v"(s), "i"(M));
}

// x_j *= dg_j, then x_r += x_j S[j][r] for r > j, 16 elements
__device__ __forceinline__ void unit_solve(float (&x)[4], const float (&S)[16], float dg) {
    static_for<0, 15>([&](auto jc) {
        constexpr int j = jc.value;
        float m[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) m[k] = row_bcast<j>(x[k] * dg);
        fma_in<above(j)>(x, m, S[j]);
    });
#pragma unroll
    for (int k = 0; k < 4; ++k) x[k] *= dg;
}

__global__ __launch_bounds__(128) void prep_kernel(const float* __restrict__ A, int64_t lda,
                                                   int64_t off, int B, float* __restrict__ DT,
                                                   float* __restrict__ inv, int64_t inv_stride,
                                                   float* pf, float* pb, int64_t words,
                                                   int* status) {
    __shared__ __attribute__((aligned(16))) float S[32][36];
    const int NQ = B / 32;
    const int t = threadIdx.x;
    int blk = blockIdx.x;
    const float* D = A + off * lda + off;
    inv += (int64_t)blockIdx.y * inv_stride;
    if (gridDim.y > 1) D += (int64_t)blockIdx.y * (B * lda + B);  // all-blocks mode
    if (pf)
        gesl_clear(pf, pb, words, status,
                   ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * 128 + t,
                   (int64_t)gridDim.x * gridDim.y * 128);
    // a 32 x 32 sub-block into S (rows are 16-byte aligned: off is a multiple
    // of 32, lda of 4)
    auto load_sub = [&](int r0, int c0) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            const int e = t + 128 * k, i = e / 8, j = (e % 8) * 4;
            *reinterpret_cast<float4*>(&S[i][j]) =
                *reinterpret_cast<const float4*>(D + (int64_t)(r0 + i) * lda + c0 + j);
        }
    };
    if (blk >= 2 * NQ) {
        blk -= 2 * NQ;
        const int tr = blk / NQ, tc = blk % NQ;
        load_sub(tr * 32, tc * 32);
        __syncthreads();
        for (int e = t; e < 1024; e += 128) {
            const int j = e / 32, i = e % 32;
            DT[(int64_t)(tc * 32 + j) * B + tr * 32 + i] = S[i][j];
        }
        return;
    }
    const bool top = blk < NQ;
    const int q = top ? blk : blk - NQ;
    load_sub(q * 32, q * 32);
    __syncthreads();
    // (w for the whole wave, so that its branches are scalar ones)
    const int r = t & 15, g = (t >> 4) & 3, w = __builtin_amdgcn_readfirstlane(t >> 6);
    // coefficients S[j][r]: top D[r][j], left D[j][r]
    auto coeff = [&](float (&s)[16], int j0, int r0) {
        if (top) {
#pragma unroll
            for (int j = 0; j < 16; j += 4) {
                const float4 v = *reinterpret_cast<const float4*>(&S[r0 + r][j0 + j]);
                s[j] = v.x;
                s[j + 1] = v.y;
                s[j + 2] = v.z;
                s[j + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int j = 0; j < 16; ++j) s[j] = S[j0 + j][r0 + r];
        }
    };
    float lo[4] = {0, 0, 0, 0}, hi[4], s[16];
    if (w == 0) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            lo[k] = 4 * g + k == r ? 1.0f : 0.0f;
            hi[k] = 0.0f;
        }
        coeff(s, 0, 0);
        unit_solve(lo, s, top ? S[r][r] : 1.0f);
        coeff(s, 0, 16);
        static_for<0, 16>([&](auto jc) {
            constexpr int j = jc.value;
#pragma unroll
            for (int k = 0; k < 4; ++k) hi[k] = fmaf(row_bcast<j>(lo[k]), s[j], hi[k]);
        });
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) hi[k] = 4 * g + k == r ? 1.0f : 0.0f;
    }
    coeff(s, 16, 16);
    unit_solve(hi, s, top ? S[16 + r][16 + r] : 1.0f);
    // out[c][i] = element i of vector c
    float* o = inv + (int64_t)(top ? q : NQ + q) * 1024 + (16 * w + 4 * g) * 32 + r;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        o[k * 32] = lo[k];
        o[k * 32 + 16] = hi[k];
    }
    if (top) {
        float* h = inv + (int64_t)(2 * NQ + q) * 1024 + r * 32 + 16 * w + 4 * g;
        *reinterpret_cast<float4*>(h) = float4{-lo[0], -lo[1], -lo[2], -lo[3]};
        *reinterpret_cast<float4*>(h + 16 * 32) = float4{-hi[0], -hi[1], -hi[2], -hi[3]};
    }
}

// ----------------------------------------------------------------------------
// The solve.  Launch: one wave per workgroup, grid.x = ceil(m/32) vectors
// groups for the top strip followed by the same count for the left strip.
// ----------------------------------------------------------------------------
// LP: element type of the optional low-precision copies for the mixed
// precision trailing update (float = none): lpT[c][k] (top strip, column c)
// and lpL[r][k] (left strip, row r), k-contiguous with leading dimension ldlp.
template <int B, typename LP>
__global__ __launch_bounds__(64) void trsm_kernel(float* __restrict__ A, int64_t lda, int64_t off,
                                                  int64_t m, const float* __restrict__ DT, int64_t lddt,
                                                  const float* __restrict__ inv, int64_t inv_ts,
                                                  float* __restrict__ Lt, int64_t ldt,
                                                  int ngroups_top, LP* __restrict__ lpT,
                                                  LP* __restrict__ lpL, int64_t ldlp,
                                                  float* __restrict__ scT,
                                                  float* __restrict__ scL) {
    constexpr bool kFp8 = std::is_same<LP, fp8e4m3>::value;
    constexpr int NQ = B / 32;
    __shared__ float Y[B][32];
    __shared__ float SZ[32][33];  // staging tile of the left strip, then z_q
    auto& Stg = SZ;
    auto& Z = SZ;
    const int lane = threadIdx.x;
    const int lr = lane & 31, lh = lane >> 5;
    const bool top = (int)blockIdx.x < ngroups_top;
    const int64_t v0 = (int64_t)(top ? blockIdx.x : blockIdx.x - ngroups_top) * 32;
    const float* D = A + off * lda + off;
    // coefficient matrix read as X[p][i]: top -> D^T, left -> D
    const float* Xc = top ? DT : D;
    const int64_t ldx = top ? lddt : lda;
    const float* G = inv + (top ? 0 : inv_ts);
    float* stripT = A + off * lda + off + B;          // top strip: rows off.., cols off+B..
    float* stripL = A + (off + B) * lda + off;        // left strip: rows off+B.., cols off..

    // prefetch of the next block's right-hand sides (registers)
    float vn[16];
    f32x4 sn[4];
    auto fetch_v = [&](int q) {
        if (top) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                vn[r] = stripT[(int64_t)(q * 32 + acc_row(r, lane)) * lda + v0 + lr];
        } else {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int vr = (lane >> 3) + 8 * s, c4 = (lane & 7) * 4;
                sn[s] = *reinterpret_cast<const f32x4*>(stripL + (v0 + vr) * lda + q * 32 + c4);
            }
        }
    };
    fetch_v(0);

    constexpr int PF = 8;  // coefficient prefetch depth (k-pairs)
    for (int q = 0; q < NQ; ++q) {
        f32x16 acc;
        // ---- v_q in accumulator layout (row i = acc_row, vector = lr)
        if (top) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[r] = vn[r];
        } else {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int vr = (lane >> 3) + 8 * s, c4 = (lane & 7) * 4;
                Stg[vr][c4 + 0] = sn[s][0];
                Stg[vr][c4 + 1] = sn[s][1];
                Stg[vr][c4 + 2] = sn[s][2];
                Stg[vr][c4 + 3] = sn[s][3];
            }
            wave_lds_sync();
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[r] = Stg[lr][acc_row(r, lane)];
        }
        if (q + 1 < NQ) fetch_v(q + 1);
        // inverse of the diagonal sub-system, loaded early
        const float* Gq = G + q * 1024;
        float g[16];
#pragma unroll
        for (int kp = 0; kp < 16; ++kp) g[kp] = Gq[(2 * kp + lh) * 32 + lr];
        // ---- z_q = v_q + C[q rows][0:32q] * Y[0:32q]   (16q k-pairs)
        const int cnt = 16 * q;
        const float* xc = Xc + (int64_t)lh * ldx + q * 32 + lr;
        float an[PF];
#pragma unroll
        for (int j = 0; j < PF; ++j) an[j] = (j < cnt) ? xc[(int64_t)(2 * j) * ldx] : 0.0f;
        for (int kp = 0; kp < cnt; kp += PF) {
            float ac[PF];
#pragma unroll
            for (int j = 0; j < PF; ++j) ac[j] = an[j];
#pragma unroll
            for (int j = 0; j < PF; ++j) {
                const int kn = kp + PF + j;
                if (kn < cnt) an[j] = xc[(int64_t)(2 * kn) * ldx];
            }
#pragma unroll
            for (int j = 0; j < PF; ++j) acc = mfma32(ac[j], Y[2 * (kp + j) + lh][lr], acc);
        }
        // ---- y_q = G_q z_q
        wave_lds_sync();  // staging reads done before z overwrites the tile
#pragma unroll
        for (int r = 0; r < 16; ++r) Z[acc_row(r, lane)][lr] = acc[r];
        wave_lds_sync();
        f32x16 y = {0};
#pragma unroll
        for (int kp = 0; kp < 16; ++kp) y = mfma32(g[kp], Z[2 * kp + lh][lr], y);
#pragma unroll
        for (int r = 0; r < 16; ++r) Y[q * 32 + acc_row(r, lane)][lr] = y[r];
        // ---- low-precision copy: registers 4g..4g+3 are 4 consecutive k
        if constexpr (!std::is_same<LP, float>::value && !kFp8) {
            LP* dst = (top ? lpT : lpL) + (v0 + lr) * ldlp + q * 32 + 4 * lh;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                struct alignas(8) P4 { LP v[4]; } p4;
#pragma unroll
                for (int e = 0; e < 4; ++e) p4.v[e] = static_cast<LP>(y[4 * g + e]);
                *reinterpret_cast<P4*>(dst + 8 * g) = p4;
            }
        }
        // ---- write back
        if (top) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                stripT[(int64_t)(q * 32 + acc_row(r, lane)) * lda + v0 + lr] = y[r];
        } else {
            if (Lt)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    Lt[(int64_t)(q * 32 + acc_row(r, lane)) * ldt + v0 + lr] = y[r];
            wave_lds_sync();
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int vr = (lane >> 3) + 8 * s, c4 = (lane & 7) * 4;
                f32x4 v;
                v[0] = Y[q * 32 + c4 + 0][vr];
                v[1] = Y[q * 32 + c4 + 1][vr];
                v[2] = Y[q * 32 + c4 + 2][vr];
                v[3] = Y[q * 32 + c4 + 3][vr];
                *reinterpret_cast<f32x4*>(stripL + (v0 + vr) * lda + q * 32 + c4) = v;
            }
        }
        wave_lds_sync();
    }
    // ---- FP8 copy with one power-of-two scale per block of 32 vectors x B:
    // lane (lr, lh) quantises vector lr, k in [lh B/2, (lh+1) B/2)
    if constexpr (kFp8) {
        constexpr int KH = B / 2;
        float am = 0.0f;
#pragma unroll 8
        for (int k = lh * KH; k < (lh + 1) * KH; ++k) am = fmaxf(am, fabsf(Y[k][lr]));
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) am = fmaxf(am, __shfl_xor(am, o));
        const int e = fp8_scale_exp(am);
        const float inv = exp2i(-e);
        uint8_t* dst = reinterpret_cast<uint8_t*>(top ? lpT : lpL) + (v0 + lr) * ldlp + lh * KH;
#pragma unroll
        for (int c = 0; c < KH; c += 16) {
            uint32_t w[4];
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                const int k = lh * KH + c + 4 * q4;
                w[q4] = fp8_e4m3_code(Y[k][lr] * inv) | (fp8_e4m3_code(Y[k + 1][lr] * inv) << 8) |
                        (fp8_e4m3_code(Y[k + 2][lr] * inv) << 16) |
                        (fp8_e4m3_code(Y[k + 3][lr] * inv) << 24);
            }
            *reinterpret_cast<uint4*>(dst + c) = make_uint4(w[0], w[1], w[2], w[3]);
        }
        if (lane == 0) (top ? scT : scL)[v0 / 32] = exp2i(e);
    }
}

// ----------------------------------------------------------------------------
// The same solve with the solved blocks kept in registers (B <= 256): no LDS
// for Y, so the kernel fits beside the trailing-update GEMM on a CU (the LDS
// version needs B*32*4 bytes per wave).  The k order of each MFMA pair
// follows the accumulator layout: register r of a lane holds row acc_row(r)
// of its block, so the lane supplies that row's y as the B operand and the
// matching coefficient as the A operand -- both z = v + C y and y = G z are
// computed from registers.
template <int B, typename LP>
__global__ __launch_bounds__(64) void trsm_reg_kernel(float* __restrict__ A, int64_t lda,
                                                      int64_t off, int64_t m,
                                                      const float* __restrict__ DT, int64_t lddt,
                                                      const float* __restrict__ inv, int64_t inv_ts,
                                                      float* __restrict__ Lt, int64_t ldt,
                                                      int ngroups_top, LP* __restrict__ lpT,
                                                      LP* __restrict__ lpL, int64_t ldlp,
                                                      float* __restrict__ scT,
                                                      float* __restrict__ scL) {
    constexpr int NQ = B / 32;
    constexpr bool kFp8 = std::is_same<LP, fp8e4m3>::value;
    constexpr bool kLp = !std::is_same<LP, float>::value && !kFp8;
    __shared__ float Tt[32][33];  // transposes of the left strip
    const int lane = threadIdx.x;
    const int lr = lane & 31;
    const bool top = (int)blockIdx.x < ngroups_top;
    const int64_t v0 = (int64_t)(top ? blockIdx.x : blockIdx.x - ngroups_top) * 32;
    const float* D = A + off * lda + off;
    const float* Xc = top ? DT : D;  // coefficients read as X[p][i]
    const int64_t ldx = top ? lddt : lda;
    const float* G = inv + (top ? 0 : inv_ts);
    float* stripT = A + off * lda + off + B;
    float* stripL = A + (off + B) * lda + off;

    f32x16 Y[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        f32x16 acc;
        if (top) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                acc[r] = stripT[(int64_t)(q * 32 + acc_row(r, lane)) * lda + v0 + lr];
        } else {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int vr = (lane >> 3) + 8 * s, c4 = (lane & 7) * 4;
                const f32x4 v =
                    *reinterpret_cast<const f32x4*>(stripL + (v0 + vr) * lda + q * 32 + c4);
                Tt[vr][c4 + 0] = v[0];
                Tt[vr][c4 + 1] = v[1];
                Tt[vr][c4 + 2] = v[2];
                Tt[vr][c4 + 3] = v[3];
            }
            wave_lds_sync();
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[r] = Tt[lr][acc_row(r, lane)];
            wave_lds_sync();
        }
        // z = v + sum over solved blocks pb < q of C[q][pb] y_pb
        float c[2][16];
        if (q > 0) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                c[0][r] = Xc[(int64_t)acc_row(r, lane) * ldx + q * 32 + lr];
        }
#pragma unroll
        for (int pb = 0; pb < q; ++pb) {
            if (pb + 1 < q) {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    c[(pb + 1) & 1][r] =
                        Xc[(int64_t)((pb + 1) * 32 + acc_row(r, lane)) * ldx + q * 32 + lr];
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) acc = mfma32(c[pb & 1][r], Y[pb][r], acc);
        }
        // y = G_q z  (G[i][k] stored at Gq[k * 32 + i])
        const float* Gq = G + q * 1024;
        f32x16 y = {0};
#pragma unroll
        for (int r = 0; r < 16; ++r) y = mfma32(Gq[acc_row(r, lane) * 32 + lr], acc[r], y);
        Y[q] = y;
        if constexpr (kLp) {
            LP* dst = (top ? lpT : lpL) + (v0 + lr) * ldlp + q * 32 + 4 * (lane >> 5);
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                struct alignas(8) P4 { LP v[4]; } p4;
#pragma unroll
                for (int e = 0; e < 4; ++e) p4.v[e] = static_cast<LP>(y[4 * g + e]);
                *reinterpret_cast<P4*>(dst + 8 * g) = p4;
            }
        }
        if (top) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                stripT[(int64_t)(q * 32 + acc_row(r, lane)) * lda + v0 + lr] = y[r];
        } else {
            if (Lt)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    Lt[(int64_t)(q * 32 + acc_row(r, lane)) * ldt + v0 + lr] = y[r];
#pragma unroll
            for (int r = 0; r < 16; ++r) Tt[acc_row(r, lane)][lr] = y[r];
            wave_lds_sync();
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int vr = (lane >> 3) + 8 * s, c4 = (lane & 7) * 4;
                f32x4 v;
                v[0] = Tt[c4 + 0][vr];
                v[1] = Tt[c4 + 1][vr];
                v[2] = Tt[c4 + 2][vr];
                v[3] = Tt[c4 + 3][vr];
                *reinterpret_cast<f32x4*>(stripL + (v0 + vr) * lda + q * 32 + c4) = v;
            }
            wave_lds_sync();
        }
    }
    // FP8 copy: one power-of-two scale for the 32 vectors x B of this wave;
    // registers 4g..4g+3 are 4 consecutive k, stored as one 32-bit word
    if constexpr (kFp8) {
        float am = 0.0f;
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int r = 0; r < 16; ++r) am = fmaxf(am, fabsf(Y[q][r]));
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) am = fmaxf(am, __shfl_xor(am, o));
        const int e = fp8_scale_exp(am);
        const float sinv = exp2i(-e);
        uint8_t* dst = reinterpret_cast<uint8_t*>(top ? lpT : lpL) + (v0 + lr) * ldlp +
                       4 * (lane >> 5);
#pragma unroll
        for (int q = 0; q < NQ; ++q)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const uint32_t w = fp8_e4m3_code(Y[q][4 * g] * sinv) |
                                   (fp8_e4m3_code(Y[q][4 * g + 1] * sinv) << 8) |
                                   (fp8_e4m3_code(Y[q][4 * g + 2] * sinv) << 16) |
                                   (fp8_e4m3_code(Y[q][4 * g + 3] * sinv) << 24);
                *reinterpret_cast<uint32_t*>(dst + q * 32 + 8 * g) = w;
            }
        if (lane == 0) (top ? scT : scL)[v0 / 32] = exp2i(e);
    }
}

// ----------------------------------------------------------------------------
// The same solve for strips that leave most of the device idle: one workgroup
// per 32 vectors, 16 vectors to each half of it, the 32-row blocks of those
// dealt out to W waves.  As soon as block p is solved every wave updates its
// blocks beyond p by it, the next one first.
//
// Bound: the chain of B/32 blocks.  With 16 vectors a product of 32 x 32
// coefficients is 16 v_mfma_f32_16x16x4_f32 of 32 cycles, half of the chain of 32
// vectors on 32x32x2, and a block's chain holds one update and the product
// with its inverse, not an update by every block before it.
//
// Operand layout: step (t, r) of a product takes k = 16 t + 4 (lane / 16) + r,
// the row that register r of accumulator tile t holds in that lane, so a
// solved block is the next product's B operand as it stands (its own inverse)
// or as two 16-byte LDS reads (the other waves).
//
// GEFA: n = 1024 B = 128 0.378 -> 0.324 ms, 2048 0.853 -> 0.738, 4096 B = 256
// 2.51 -> 1.94, B = 64 2.15 -> 2.00; FP8 n = 6144 B = 128 3.3 -> 2.95, B = 256
// 3.69 -> 2.86.
template <int B>
constexpr int kSplitWaves = B / 32 < 4 ? B / 32 : 4;  // per half

template <int B, typename LP>
__global__ __launch_bounds__(128 * kSplitWaves<B>) void trsm_split_kernel(
    float* __restrict__ A, int64_t lda, int64_t off, const float* DT, int64_t lddt,
    const float* __restrict__ inv, int64_t inv_ts, float* Lt, int64_t ldt, int ngroups_top,
    LP* __restrict__ lpT, LP* __restrict__ lpL, int64_t ldlp, float* __restrict__ scT,
    float* __restrict__ scL) {
    constexpr int NQ = B / 32, W = kSplitWaves<B>, NO = NQ / W;  // blocks per wave
    constexpr bool kFp8 = std::is_same<LP, fp8e4m3>::value;
    constexpr bool kLp = !std::is_same<LP, float>::value && !kFp8;
    __shared__ __attribute__((aligned(16))) float Ys[2][2][16][36];
    __shared__ float am_sh[2 * W];
    const int lane = threadIdx.x & 63, wave = (threadIdx.x >> 6) % W;
    const int half = (threadIdx.x >> 6) / W;
    const int c = lane & 15, kk = lane >> 4;
    const bool top = (int)blockIdx.x < ngroups_top;
    const int64_t g32 = top ? blockIdx.x : blockIdx.x - ngroups_top;
    const int64_t v = g32 * 32 + 16 * half + c;  // this lane's vector
    const float* G = inv + (top ? 0 : inv_ts);
    float* stripT = A + off * lda + off + B + v;
    float* stripL = A + (off + B + v) * lda + off;
    auto Y = Ys[half];

    // coefficients X[p][i] of block (q, p) for step (t2, r) and row tile t: top
    // D^T, left D
    const float* X = top ? DT : A + off * lda + off;
    const int64_t ldx = top ? lddt : lda;
    auto load_c = [&](float (&x)[2][2][4], int q, int p) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    x[t][t2][r] = X[(p * 32 + 16 * t2 + 4 * kk + r) * ldx + q * 32 + 16 * t + c];
    };
    float g[NO][2][2][4], cn[NO][2][2][4];
    f32x4 acc[NO][2];
#pragma unroll
    for (int m = 0; m < NO; ++m) {
        const int q = wave + W * m;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int64_t k = q * 32 + 16 * t + 4 * kk;
            if (top) {
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[m][t][r] = stripT[(k + r) * lda];
            } else {
                acc[m][t] = *reinterpret_cast<const f32x4*>(stripL + k);
            }
#pragma unroll
            for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    g[m][t][t2][r] = G[q * 1024 + (16 * t2 + 4 * kk + r) * 32 + 16 * t + c];
        }
        if (q > 0) load_c(cn[m], q, 0);
    }
    for (int p = 0; p < NQ; ++p) {
        if (p % W == wave) {
            // y_p = G_p z_p
            f32x4 y[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
            for (int m = 0; m < NO; ++m)
                if (p == wave + W * m) {
#pragma unroll
                    for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
#pragma unroll
                            for (int t = 0; t < 2; ++t)
                                y[t] = mfma16(g[m][t][t2][r], acc[m][t2][r], y[t]);
                    acc[m][0] = y[0];
                    acc[m][1] = y[1];
                }
#pragma unroll
            for (int t = 0; t < 2; ++t)
                *reinterpret_cast<f32x4*>(&Y[p & 1][c][16 * t + 4 * kk]) = y[t];
        }
        if (p + 1 == NQ) break;
        __syncthreads();
        f32x4 yv[2];
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2)
            yv[t2] = *reinterpret_cast<const f32x4*>(&Y[p & 1][c][16 * t2 + 4 * kk]);
#pragma unroll
        for (int m = 0; m < NO; ++m) {
            const int q = wave + W * m;
            if (q > p) {
                float x[2][2][4];
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
                        for (int r = 0; r < 4; ++r) x[t][t2][r] = cn[m][t][t2][r];
                if (q > p + 1) load_c(cn[m], q, p + 1);  // for the next block
#pragma unroll
                for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int t = 0; t < 2; ++t)
                            acc[m][t] = mfma16(x[t][t2][r], yv[t2][r], acc[m][t]);
            }
        }
    }
    // ---- write back: acc[m][t][r] is element 32 q + 16 t + 4 kk + r
    float sinv = 1.0f;
    if constexpr (kFp8) {
        // one power-of-two scale for the workgroup's 32 vectors x B
        float am = 0.0f;
#pragma unroll
        for (int m = 0; m < NO; ++m)
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) am = fmaxf(am, fabsf(acc[m][t][r]));
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) am = fmaxf(am, __shfl_xor(am, o));
        if (lane == 0) am_sh[threadIdx.x >> 6] = am;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < 2 * W; ++w) am = fmaxf(am, am_sh[w]);
        const int e = fp8_scale_exp(am);
        sinv = exp2i(-e);
        if (threadIdx.x == 0) (top ? scT : scL)[g32] = exp2i(e);
    }
#pragma unroll
    for (int m = 0; m < NO; ++m)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int64_t k = (wave + W * m) * 32 + 16 * t + 4 * kk;
            const f32x4 y = acc[m][t];
            if (top) {
#pragma unroll
                for (int r = 0; r < 4; ++r) stripT[(k + r) * lda] = y[r];
            } else {
                *reinterpret_cast<f32x4*>(stripL + k) = y;
                if (Lt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) Lt[(k + r) * ldt + v] = y[r];
            }
            if constexpr (kLp) {
                struct alignas(8) P4 { LP e[4]; } p4;
#pragma unroll
                for (int r = 0; r < 4; ++r) p4.e[r] = static_cast<LP>(y[r]);
                *reinterpret_cast<P4*>((top ? lpT : lpL) + v * ldlp + k) = p4;
            }
            if constexpr (kFp8) {
                uint8_t* dst = reinterpret_cast<uint8_t*>(top ? lpT : lpL) + v * ldlp + k;
                *reinterpret_cast<uint32_t*>(dst) =
                    fp8_e4m3_code(y[0] * sinv) | (fp8_e4m3_code(y[1] * sinv) << 8) |
                    (fp8_e4m3_code(y[2] * sinv) << 16) | (fp8_e4m3_code(y[3] * sinv) << 24);
            }
        }
}

// ----------------------------------------------------------------------------
// Full inverses of the diagonal blocks for the substitution.  The strip
// recurrences above, run on unit vectors, give for diagonal block k (with
// L unit lower and U upper as the substitution uses them, M terms):
//   left recurrence on e_r :  y = L^-1 e_r      -> OutL[r][i] = (L^-1)(i, r)
//   top  recurrence on e_c :  y = -(U^T)^-1 e_c -> OutU[i][c] = -(U^-1)(c, i)
// stored per block at out + k * 2 * B * B (OutL, then OutU), both row-major
// B x B, so the substitution applies them as coalesced GEMVs.  Launch: grid
// (B/16 vector groups, 2 types, blocks), four waves each; coefficients are
// read straight from the factor.
//
// Bound: the chain of B/32 blocks, per block one update by the block before
// and the product with its 32 x 32 inverse.  Wave w owns the 32-row blocks w
// and w + 4 of the group's 16 vectors; as soon as block p is solved every
// wave updates its blocks beyond p by it, the next one first.  With 16
// vectors a product of 32 x 32 coefficients is 16 v_mfma_f32_16x16x4_f32 of
// 32 cycles, half the chain of 32 vectors on 32x32x2; blocks before the unit
// vectors' own are zero and skipped.  (B = 256: 38 us with one wave solving
// all blocks of 32 vectors in turn, 13 us here; hpl_gesl_noalloc at n = 1024
// 72.3 -> 47.6 us, BF16 refinement at n = 65536 279.7 -> 278.2 ms.)
//
// Operand layout: step (t, r) of a product takes k = 16 t + 4 (lane / 16) + r,
// the row that register r of accumulator tile t holds in that lane, so a
// solved block is the next product's B operand as it stands (its own inverse)
// or as two 16-byte LDS reads (the other waves).
//
// pk, if not null: the inverses' BF16 operand copies of the strip solves
// (below), written from the same registers.
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

template <int B>
__global__ __launch_bounds__(256) void block_inverse_kernel(const float* __restrict__ A,
                                                            int64_t lda,
                                                            const float* __restrict__ inv,
                                                            int64_t inv_stride,
                                                            float* __restrict__ out,
                                                            bf16x8_t* __restrict__ pk) {
    constexpr int NQ = B / 32, NB = NQ * (NQ + 1) / 2;
    constexpr int NO = (NQ + 3) / 4;  // blocks per wave
    __shared__ __attribute__((aligned(16))) float Y[2][16][36];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = lane & 15, kk = lane >> 4;
    const int v0 = blockIdx.x * 16, vb = v0 / 32;
    const bool top = blockIdx.y == 0;
    const int64_t k = blockIdx.z;
    const float* D = A + k * B * lda + k * B;
    const float* G = inv + k * inv_stride + (top ? 0 : NQ * 1024);
    float* o = out + k * 2 * (int64_t)B * B + (top ? (int64_t)B * B : 0);
    const int64_t ostep_i = top ? B : 1, ostep_v = top ? 1 : B;  // o offset per element / vector

    // zeros above the unit vectors' block
    for (int e = threadIdx.x; e < vb * 32 * 16; e += 256) {
        const int i = top ? e / 16 : e % (vb * 32), v = top ? e % 16 : e / (vb * 32);
        o[i * ostep_i + (v0 + v) * ostep_v] = 0.0f;
    }

    // coefficients of block (q, p) for step (t2, r) and row tile t: X[p][i],
    // top D[i][p], left D[p][i]
    auto load_c = [&](float (&x)[2][2][4], int q, int p) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int t2 = 0; t2 < 2; ++t2) {
                const int64_t i = q * 32 + 16 * t + c, kp = p * 32 + 16 * t2 + 4 * kk;
                if (top) {
                    const f32x4 v = *reinterpret_cast<const f32x4*>(D + i * lda + kp);
#pragma unroll
                    for (int r = 0; r < 4; ++r) x[t][t2][r] = v[r];
                } else {
#pragma unroll
                    for (int r = 0; r < 4; ++r) x[t][t2][r] = D[(kp + r) * lda + i];
                }
            }
    };
    float g[NO][2][2][4], cn[NO][2][2][4];
    f32x4 acc[NO][2];
#pragma unroll
    for (int m = 0; m < NO; ++m) {
        const int q = wave + 4 * m;
        const bool mine = q < NQ && q >= vb;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                acc[m][t][r] = q * 32 + 16 * t + 4 * kk + r == v0 + c ? 1.0f : 0.0f;
                g[m][t][0][r] = g[m][t][1][r] = cn[m][t][0][r] = cn[m][t][1][r] = 0.0f;
            }
        if (mine) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        g[m][t][t2][r] = G[q * 1024 + (16 * t2 + 4 * kk + r) * 32 + 16 * t + c];
            if (q > vb) load_c(cn[m], q, vb);
        }
    }
    for (int p = vb; p < NQ; ++p) {
        if ((p & 3) == wave) {
            // y_p = G_p z_p
            f32x4 y[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
            for (int m = 0; m < NO; ++m)
                if (p == wave + 4 * m) {
#pragma unroll
                    for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
#pragma unroll
                            for (int t = 0; t < 2; ++t)
                                y[t] = mfma16(g[m][t][t2][r], acc[m][t2][r], y[t]);
                }
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                *reinterpret_cast<f32x4*>(&Y[p & 1][c][16 * t + 4 * kk]) = y[t];
                // element i = p*32 + 16 t + 4 kk + r of vector v0 + c
                const int64_t i = p * 32 + 16 * t + 4 * kk;
                if (top) {
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[(i + r) * B + v0 + c] = y[t][r];
                } else {
                    *reinterpret_cast<f32x4*>(o + (v0 + c) * (int64_t)B + i) = y[t];
                }
                if (pk) {
                    // operand copy: row i % 32, k = v0 + c of block (p, vb)
                    __bf16* d = reinterpret_cast<__bf16*>(
                        pk + ((top ? 0 : NB) + p * (p + 1) / 2 + vb) * (int64_t)256);
                    const int kc = (v0 & 31) + c, kb = kc >> 4, h = (kc >> 3) & 1, e = kc & 7;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int l = 16 * t + 4 * kk + r + 32 * h;
                        const __bf16 hi = static_cast<__bf16>(y[t][r]);
                        d[((kb * 2 + 0) * 64 + l) * 8 + e] = hi;
                        d[((kb * 2 + 1) * 64 + l) * 8 + e] =
                            static_cast<__bf16>(y[t][r] - static_cast<float>(hi));
                    }
                }
            }
        }
        if (p + 1 == NQ) break;
        __syncthreads();
        f32x4 yv[2];
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2)
            yv[t2] = *reinterpret_cast<const f32x4*>(&Y[p & 1][c][16 * t2 + 4 * kk]);
#pragma unroll
        for (int m = 0; m < NO; ++m) {
            const int q = wave + 4 * m;
            if (q > p && q < NQ) {
                float x[2][2][4];
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
                        for (int r = 0; r < 4; ++r) x[t][t2][r] = cn[m][t][t2][r];
                if (q > p + 1) load_c(cn[m], q, p + 1);  // for the next block
#pragma unroll
                for (int t2 = 0; t2 < 2; ++t2)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
#pragma unroll
                        for (int t = 0; t < 2; ++t)
                            acc[m][t] = mfma16(x[t][t2][r], yv[t2][r], acc[m][t]);
            }
        }
    }
}

// ----------------------------------------------------------------------------
// Strip solves of the BF16 factorisation as products with the diagonal
// block's full inverses.  The top and left recurrences above are linear maps
// y = G v with G lower triangular (G_top = OutU, G_left = OutL transposed, as
// block_inverse_kernel writes them), so each strip is one product over
// independent 32 x 32 blocks, y_q = sum_{p <= q} G_qp v_p: no chain from block
// to block, every load of v issued before the first MFMA.  The product runs on
// v_mfma_f32_32x32x16_bf16 with each operand split as x = hi + lo (hi =
// bf16(x), lo = bf16(x - hi), both exact to about 2^-17 |x|) and
// G v = G_hi v_hi + G_hi v_lo + G_lo v_hi.
//
// Operand layout of one 32 x 32 block product (two MFMAs of K = 16): lane
// (i, h) = (l % 32, l / 32) supplies G[i][16 kb + 8 h + e] and, for vector
// i, v[16 kb + 8 h + e], e = 0..7.  block_inverse_kernel writes G in that layout
// once per step: block (q, p), p <= q, at index q (q + 1) / 2 + p, 2048
// halves each -- [kb][hi, lo][lane][8].
__device__ __forceinline__ void split_bf16(const float (&x)[8], bf16x8_t& hi, bf16x8_t& lo) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const __bf16 h = static_cast<__bf16>(x[e]);
        hi[e] = h;
        lo[e] = static_cast<__bf16>(x[e] - static_cast<float>(h));
    }
}

// One wave per 32 vectors: grid.x = ngroups_top top groups, then as many left
// groups.
template <int B, typename LP>
__global__ __launch_bounds__(64) void trsm_inv_kernel(float* __restrict__ A, int64_t lda,
                                                      int64_t off,
                                                      const bf16x8_t* __restrict__ pk,
                                                      int ngroups_top, LP* __restrict__ lpT,
                                                      LP* __restrict__ lpL, int64_t ldlp) {
    constexpr int NQ = B / 32, NB = NQ * (NQ + 1) / 2;
    const int lane = threadIdx.x;
    const int lr = lane & 31, lh = lane >> 5;
    const bool top = (int)blockIdx.x < ngroups_top;
    const int64_t v0 = (int64_t)(top ? blockIdx.x : blockIdx.x - ngroups_top) * 32;
    float* stripT = A + off * lda + off + B;
    float* stripL = A + (off + B) * lda + off;
    const bf16x8_t* G = pk + (top ? 0 : NB * 256) + lane;

    // v of vector v0 + lr, k = 32 p + 16 kb + 8 lh + e, split into halves
    bf16x8_t vh[NQ][2], vl[NQ][2];
    {
        float x[NQ][2][8];
#pragma unroll
        for (int p = 0; p < NQ; ++p)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                const int k0 = p * 32 + 16 * kb + 8 * lh;
                if (top) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) x[p][kb][e] = stripT[(int64_t)(k0 + e) * lda + v0 + lr];
                } else {
                    const float* src = stripL + (v0 + lr) * lda + k0;
                    const f32x4 a = *reinterpret_cast<const f32x4*>(src);
                    const f32x4 b = *reinterpret_cast<const f32x4*>(src + 4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        x[p][kb][e] = a[e];
                        x[p][kb][4 + e] = b[e];
                    }
                }
            }
#pragma unroll
        for (int p = 0; p < NQ; ++p)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) split_bf16(x[p][kb], vh[p][kb], vl[p][kb]);
    }

#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        f32x16 acc = {0};
#pragma unroll
        for (int p = 0; p <= q; ++p) {
            const bf16x8_t* g = G + (int64_t)(q * (q + 1) / 2 + p) * 256;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                const bf16x8_t ghi = g[(kb * 2 + 0) * 64], glo = g[(kb * 2 + 1) * 64];
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(glo, vh[p][kb], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ghi, vl[p][kb], acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ghi, vh[p][kb], acc, 0, 0, 0);
            }
        }
        // register r: element i = q * 32 + acc_row(r) of vector v0 + lr
        LP* dst = (top ? lpT : lpL) + (v0 + lr) * ldlp + q * 32 + 4 * lh;
#pragma unroll
        for (int g4 = 0; g4 < 4; ++g4) {
            struct alignas(8) P4 {
                LP v[4];
            } p4;
#pragma unroll
            for (int e = 0; e < 4; ++e) p4.v[e] = static_cast<LP>(acc[4 * g4 + e]);
            *reinterpret_cast<P4*>(dst + 8 * g4) = p4;
        }
        if (top) {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                stripT[(int64_t)(q * 32 + acc_row(r, lane)) * lda + v0 + lr] = acc[r];
        } else {
            float* row = stripL + (v0 + lr) * lda + q * 32 + 4 * lh;
#pragma unroll
            for (int g4 = 0; g4 < 4; ++g4) {
                f32x4 v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = acc[4 * g4 + e];
                *reinterpret_cast<f32x4*>(row + 8 * g4) = v;
            }
        }
    }
}

}  // namespace

static hipError_t block_inverse(dim3 grid, const float* A, int64_t lda, int B, const float* inv,
                                int64_t inv_stride, float* out, bf16x8_t* pk, hipStream_t s) {
    // 16-byte row vectors
    if ((lda & 3) || (reinterpret_cast<uintptr_t>(A) & 15) ||
        (reinterpret_cast<uintptr_t>(out) & 15))
        return hipErrorInvalidValue;
    switch (B) {
#define HPL_BINV(BB)                                                                   \
    case BB:                                                                           \
        block_inverse_kernel<BB><<<grid, 256, 0, s>>>(A, lda, inv, inv_stride, out, pk); \
        break;
        HPL_BINV(32)
        HPL_BINV(64)
        HPL_BINV(128)
        HPL_BINV(256)
#undef HPL_BINV
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_block_inverse(const float* A, int64_t lda, int64_t n, int B, const float* inv,
                                int64_t inv_stride, float* out, hipStream_t s) {
    if (n % B) return hipErrorInvalidValue;
    dim3 grid(B / 16, 2, (unsigned)(n / B));
    return block_inverse(grid, A, lda, B, inv, inv_stride, out, nullptr, s);
}

hipError_t launch_prep(const float* A, int64_t lda, int64_t off, int B, float* DT, float* inv,
                       hipStream_t s) {
    if ((lda & 3) || (off & 3) || (reinterpret_cast<uintptr_t>(A) & 15))
        return hipErrorInvalidValue;  // 16-byte row vectors
    const int NQ = B / 32;
    dim3 grid(2 * NQ + (DT ? NQ * NQ : 0), 1);
    prep_kernel<<<grid, 128, 0, s>>>(A, lda, off, B, DT, inv, 0, nullptr, nullptr, 0,
                                     nullptr);
    return hipGetLastError();
}

hipError_t launch_prep_all(const float* A, int64_t lda, int B, int nblocks, float* inv,
                           int64_t inv_stride, hipStream_t s, const GeslWs* ws) {
    if ((lda & 3) || (reinterpret_cast<uintptr_t>(A) & 15)) return hipErrorInvalidValue;
    const int NQ = B / 32;
    dim3 grid(2 * NQ, nblocks);
    prep_kernel<<<grid, 128, 0, s>>>(A, lda, 0, B, nullptr, inv, inv_stride,
                                     ws ? ws->pf : nullptr, ws ? ws->pb : nullptr,
                                     gesl_ws_words((int64_t)nblocks * B, B),
                                     ws ? ws->status : nullptr);
    return hipGetLastError();
}

// Strips of up to this many vectors a side take trsm_split_kernel: 16 waves of
// registers per 64 vectors where trsm_reg_kernel has two, which beside a large
// update costs more than the shorter chain gives (GEFA n = 32768, B = 256, all
// steps by it 201.1 ms, none 198.6, up to 12288 196.7; n = 16384 29.2, none 30.5).
constexpr int64_t kSplitStrips = 12288;

// ... where the left strip's 16-byte vectors are aligned
static bool split_ok(const float* A, int64_t lda, int64_t off, int64_t m, int64_t ldlp) {
    return m <= kSplitStrips && !(lda & 3) && !(off & 3) && !(ldlp & 3) &&
           !(reinterpret_cast<uintptr_t>(A) & 15);
}

template <typename LP>
static hipError_t launch_trsm_t(float* A, int64_t lda, int64_t off, int64_t m, int B,
                                const float* DT, int64_t lddt, const float* inv, int64_t inv_ts,
                                float* Lt, int64_t ldt, LP* lpT, LP* lpL, int64_t ldlp, hipStream_t s,
                                float* scT = nullptr, float* scL = nullptr) {
    const int groups = (int)(m / 32);
    dim3 grid(2 * groups);
    if (split_ok(A, lda, off, m, ldlp)) {
#define HPL_TRSM_SPLIT(BB)                                                                    \
    case BB:                                                                                  \
        trsm_split_kernel<BB, LP><<<grid, 128 * kSplitWaves<BB>, 0, s>>>(                     \
            A, lda, off, DT, lddt, inv, inv_ts, Lt, ldt, groups, lpT, lpL, ldlp, scT, scL);   \
        return hipGetLastError();
        switch (B) {
            HPL_TRSM_SPLIT(64)
            HPL_TRSM_SPLIT(128)
            HPL_TRSM_SPLIT(256)
            default: break;
        }
#undef HPL_TRSM_SPLIT
    }
#define HPL_TRSM_CASE(BB, KERNEL)                                                             \
    case BB:                                                                                  \
        KERNEL<BB, LP><<<grid, 64, 0, s>>>(A, lda, off, m, DT, lddt, inv, inv_ts, Lt, ldt, groups, \
                                           lpT, lpL, ldlp, scT, scL);                         \
        break;
    switch (B) {
        HPL_TRSM_CASE(32, trsm_reg_kernel)
        HPL_TRSM_CASE(64, trsm_reg_kernel)
        HPL_TRSM_CASE(128, trsm_reg_kernel)
        HPL_TRSM_CASE(256, trsm_reg_kernel)
        HPL_TRSM_CASE(512, trsm_kernel)
        default: return hipErrorInvalidValue;
    }
#undef HPL_TRSM_CASE
    return hipGetLastError();
}

hipError_t launch_trsm_top(float* A, int64_t lda, int64_t off, int64_t m, int B, const float* DT,
                           const float* inv, hipStream_t s) {
    if (m <= 0) return hipSuccess;
    if (m % 32) return hipErrorInvalidValue;
    const int groups = (int)(m / 32);
    // (not trsm_split_kernel: beside the other stream's update its workgroups
    // wait longer than they gain, n = 6144 25.8 ms against 25.5)
#define HPL_TRSM_TOP(BB)                                                                      \
    case BB:                                                                                  \
        trsm_reg_kernel<BB, float><<<groups, 64, 0, s>>>(A, lda, off, m, DT, BB, inv,         \
                                                         (BB / 32) * 1024, nullptr, 0, groups, \
                                                         nullptr, nullptr, 0, nullptr,        \
                                                         nullptr);                            \
        break;
    switch (B) {
        HPL_TRSM_TOP(32)
        HPL_TRSM_TOP(64)
        HPL_TRSM_TOP(128)
        HPL_TRSM_TOP(256)
        default: return hipErrorInvalidValue;
    }
#undef HPL_TRSM_TOP
    return hipGetLastError();
}

hipError_t launch_trsm(float* A, int64_t lda, int64_t off, int64_t m, int B, const float* DT,
                       int64_t lddt, const float* inv, int64_t inv_ts, float* Lt, int64_t ldt, hipStream_t s, int lp_prec,
                       void* lpT, void* lpL, int64_t ldlp, float* scT, float* scL) {
    if (m <= 0) return hipSuccess;
    if (m % 32) return hipErrorInvalidValue;
    switch (lp_prec) {
        case 0:
            return launch_trsm_t<float>(A, lda, off, m, B, DT, lddt, inv, inv_ts, Lt, ldt, nullptr, nullptr, 0, s);
        case 1:
            return launch_trsm_t<__bf16>(A, lda, off, m, B, DT, lddt, inv, inv_ts, Lt, ldt,
                                         static_cast<__bf16*>(lpT), static_cast<__bf16*>(lpL),
                                         ldlp, s);
        case 2:
            return launch_trsm_t<_Float16>(A, lda, off, m, B, DT, lddt, inv, inv_ts, Lt, ldt,
                                           static_cast<_Float16*>(lpT),
                                           static_cast<_Float16*>(lpL), ldlp, s);
        case 3:
            if (!scT || !scL || ldlp % 16) return hipErrorInvalidValue;
            return launch_trsm_t<fp8e4m3>(A, lda, off, m, B, DT, lddt, inv, inv_ts, Lt, ldt,
                                          static_cast<fp8e4m3*>(lpT), static_cast<fp8e4m3*>(lpL),
                                          ldlp, s, scT, scL);
        default:
            return hipErrorInvalidValue;
    }
}

int64_t tinv_floats(int B) {
    const int NQ = B / 32;
    // OutL and OutU, then the packed halves (2048 per block, 2 bytes each)
    return 2 * (int64_t)B * B + (int64_t)NQ * (NQ + 1) * 2048 / 2;
}

hipError_t launch_tinv_prepare(const float* A, int64_t lda, int64_t off, int B, const float* inv,
                               float* tinv, float* out, hipStream_t s) {
    if (B % 32 || B > 256 || B < 32 || (reinterpret_cast<uintptr_t>(tinv) & 15))
        return hipErrorInvalidValue;
    bf16x8_t* pk = reinterpret_cast<bf16x8_t*>(tinv + 2 * (int64_t)B * B);
    return block_inverse(dim3(B / 16, 2, 1), A + off * lda + off, lda, B, inv, 0,
                         out ? out : tinv, pk, s);
}

hipError_t launch_trsm_inv(float* A, int64_t lda, int64_t off, int64_t m, int B,
                           const float* tinv, hipStream_t s, int lp_prec, void* lpT, void* lpL,
                           int64_t ldlp) {
    if (m <= 0) return hipSuccess;
    if (m % 32 || (lda & 3) || (off & 3) || (ldlp & 3) || (lp_prec != 1 && lp_prec != 2))
        return hipErrorInvalidValue;
    const int groups = (int)(m / 32);
    const bf16x8_t* pk = reinterpret_cast<const bf16x8_t*>(tinv + 2 * (int64_t)B * B);
    dim3 grid(2 * groups);
#define HPL_TRSM_INV(BB)                                                                      \
    case BB:                                                                                  \
        if (lp_prec == 1)                                                                     \
            trsm_inv_kernel<BB, __bf16><<<grid, 64, 0, s>>>(A, lda, off, pk, groups,           \
                                                            static_cast<__bf16*>(lpT),         \
                                                            static_cast<__bf16*>(lpL), ldlp);  \
        else                                                                                  \
            trsm_inv_kernel<BB, _Float16><<<grid, 64, 0, s>>>(A, lda, off, pk, groups,         \
                                                              static_cast<_Float16*>(lpT),     \
                                                              static_cast<_Float16*>(lpL),     \
                                                              ldlp);                           \
        break;
    switch (B) {
        HPL_TRSM_INV(32)
        HPL_TRSM_INV(64)
        HPL_TRSM_INV(128)
        HPL_TRSM_INV(256)
        default: return hipErrorInvalidValue;
    }
#undef HPL_TRSM_INV
    return hipGetLastError();
}
