// Diagonal-block LU ("lu", LINPACK/src/device/hpl_torus_PCIE.cl:211-446) and
// the 32 x 32 inverses that the strip solves and the substitution apply.
//
// Factorises the B x B diagonal block D = A[off.., off..] (row-major, lda) in
// place into the dgefa encoding without pivoting, i.e. gefa_ref_nopvt on the
// block (LINPACK/src/host/linpack_data.cpp:166-196):
//   for gk: D[gk][gk] = -1/D[gk][gk]; D[gk][c] *= D[gk][gk] (c > gk);
//           D[r][c] += D[gk][c] * D[r][gk]  (r > gk, c > gk).
// Every element receives the same multiplies and adds in the same order as in
// the reference loop (no FMA contraction), so the result is bit-identical.
//
// One workgroup; the block lives in LDS and is processed in panels of 16
// pivot rows, two stages per panel:
//   1. wave 0 applies the previous panel's rank-16 update to the panel's 16 x 16
//      diagonal sub-block and factorises it in registers.  The other waves apply
//      that update to the rest, carry on the solves of the unit vectors that
//      give the inverses, and in the last half of the panels store what is
//      finished.
//   2. every column right of the sub-block (top strip) and every row below it
//      (left strip) is solved against the sub-block, 16 vectors per wave.
// So the chain from pivot to pivot holds one 16 x 16 update, one factorisation
// and one 16-step solve per panel, not the whole trailing update.
//
// Bound: the instructions of one wave, of which one issues every 6 to 8 cycles
// whether the next depends on it or not: a pivot step of stage 1 is 25 of them
// (168 cycles), a step of stage 2 15 (100).  Hence 16-wide panels (a step of a
// 32-wide one took 45 and 320 cycles): the columns of a sub-block lie in the 16
// lanes of a DPP row, so that a multiplier is broadcast within the multiply
// (row_newbcast) and needs neither LDS nor an instruction of its own; the
// strips have an element of their vectors per lane for the same reason.  Masks
// are immediates of the exec register, one change for all rows of a step.  The
// scaled rows stay in registers of their own beside the multipliers and are
// put together once per panel.
// A tile of the trailing update is 4000 to 5000 cycles of one wave, also when it
// is alone on its SIMD, so B = 128 takes 16 waves: with 8, 35.4 us.  Panels 1
// and 2 are still bound by that update (8300 and 6400 cycles of stage 1, 3700
// the others).
// Alone on the device, with the inverses and DT: B = 128 31.9 us (32-wide
// panels 39.6; one stage at a time 62.2 and a further launch of 8 for the
// inverses), B = 64 14.4 (21.3; 26.1 + 8), B = 32 8.9 (11.0; 9.2 + 7).  GEFA at
// B = 128: n = 1024 0.454 -> 0.379 ms, 2048 1.008 -> 0.860, 4096 2.43 -> 2.12;
// B = 64 n = 7488 6.75 -> 6.0.
// With 8 waves at most 128 VGPRs and 77 KiB of LDS: the workgroup fits into
// what one of the two workgroups of the FP32 trailing update on a CU leaves.
// Blocks up to 128 are handled here; larger diagonal blocks are factorised by
// the host schedule as a 2 x 2 recursion on top of this kernel.
#include "common.hpp"
#include "kernels.hpp"

namespace {

__device__ __forceinline__ float bcast(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// d[i] += m[i], i < N, in the lanes that the mask M has in each half of the wave:
// one change of the exec mask instead of a select per value (every lane of the
// wave is active here).  The compiler does not look into the text: d is written
// before all of m is read (+&), and a DPP move may follow at once, which needs two
// wait states after the last sum -- the move to exec is one, s_nop 0 the other.
template <unsigned M, int N>
__device__ __forceinline__ void add_in(float* d, const float* m) {
    static_assert(N >= 1 && N <= 8, "up to eight values");
    if constexpr (N == 1)
        asm("s_mov_b32 exec_lo, %2\n\ts_mov_b32 exec_hi, %2\n\t"
            "v_add_f32 %0, %0, %1\n\t"
            "s_mov_b64 exec, -1\n\ts_nop 0"
            : "+&v"(d[0])
            : "v"(m[0]), "i"(M));
    else if constexpr (N == 2)
        asm("s_mov_b32 exec_lo, %4\n\ts_mov_b32 exec_hi, %4\n\t"
            "v_add_f32 %0, %0, %2\n\tv_add_f32 %1, %1, %3\n\t"
            "s_mov_b64 exec, -1\n\ts_nop 0"
            : "+&v"(d[0]), "+&v"(d[1])
            : "v"(m[0]), "v"(m[1]), "i"(M));
    else if constexpr (N == 3)
        asm("s_mov_b32 exec_lo, %6\n\ts_mov_b32 exec_hi, %6\n\t"
            "v_add_f32 %0, %0, %3\n\tv_add_f32 %1, %1, %4\n\t"
            "v_add_f32 %2, %2, %5\n\t"
            "s_mov_b64 exec, -1\n\ts_nop 0"
            : "+&v"(d[0]), "+&v"(d[1]), "+&v"(d[2])
            : "v"(m[0]), "v"(m[1]), "v"(m[2]), "i"(M));
    else if constexpr (N == 4)
        asm("s_mov_b32 exec_lo, %8\n\ts_mov_b32 exec_hi, %8\n\t"
            "v_add_f32 %0, %0, %4\n\tv_add_f32 %1, %1, %5\n\t"
            "v_add_f32 %2, %2, %6\n\tv_add_f32 %3, %3, %7\n\t"
            "s_mov_b64 exec, -1\n\ts_nop 0"
            : "+&v"(d[0]), "+&v"(d[1]), "+&v"(d[2]), "+&v"(d[3])
            : "v"(m[0]), "v"(m[1]), "v"(m[2]), "v"(m[3]), "i"(M));
    else if constexpr (N == 5)
        asm("s_mov_b32 exec_lo, %10\n\ts_mov_b32 exec_hi, %10\n\t"
            "v_add_f32 %0, %0, %5\n\tv_add_f32 %1, %1, %6\n\t"
            "v_add_f32 %2, %2, %7\n\tv_add_f32 %3, %3, %8\n\t"
            "v_add_f32 %4, %4, %9\n\t"
            "s_mov_b64 exec, -1\n\ts_nop 0"
            : "+&v"(d[0]), "+&v"(d[1]), "+&v"(d[2]), "+&v"(d[3]), "+&v"(d[4])
            : "v"(m[0]), "v"(m[1]), "v"(m[2]), "v"(m[3]), "v"(m[4]), "i"(M));
    else if constexpr (N == 6)
        asm("s_mov_b32 exec_lo, %12\n\ts_mov_b32 exec_hi, %12\n\t"
            "v_add_f32 %0, %0, %6\n\tv_add_f32 %1, %1, %7\n\t"
            "v_add_f32 %2, %2, %8\n\tv_add_f32 %3, %3, %9\n\t"
            "v_add_f32 %4, %4, %10\n\tv_add_f32 %5, %5, %11\n\t"
            "s_mov_b64 exec, -1\n\ts_nop 0"
            : "+&v"(d[0]), "+&v"(d[1]), "+&v"(d[2]), "+&v"(d[3]), "+&v"(d[4]), "+&v"(d[5])
            : "v"(m[0]), "v"(m[1]), "v"(m[2]), "v"(m[3]), "v"(m[4]), "v"(m[5]), "i"(M));
    else if constexpr (N == 7)
        asm("s_mov_b32 exec_lo, %14\n\ts_mov_b32 exec_hi, %14\n\t"
            "v_add_f32 %0, %0, %7\n\tv_add_f32 %1, %1, %8\n\t"
            "v_add_f32 %2, %2, %9\n\tv_add_f32 %3, %3, %10\n\t"
            "v_add_f32 %4, %4, %11\n\tv_add_f32 %5, %5, %12\n\t"
            "v_add_f32 %6, %6, %13\n\t"
            "s_mov_b64 exec, -1\n\ts_nop 0"
            : "+&v"(d[0]), "+&v"(d[1]), "+&v"(d[2]), "+&v"(d[3]), "+&v"(d[4]), "+&v"(d[5]), "+&v"(d[6])
            : "v"(m[0]), "v"(m[1]), "v"(m[2]), "v"(m[3]), "v"(m[4]), "v"(m[5]), "v"(m[6]), "i"(M));
    else if constexpr (N == 8)
        asm("s_mov_b32 exec_lo, %16\n\ts_mov_b32 exec_hi, %16\n\t"
            "v_add_f32 %0, %0, %8\n\tv_add_f32 %1, %1, %9\n\t"
            "v_add_f32 %2, %2, %10\n\tv_add_f32 %3, %3, %11\n\t"
            "v_add_f32 %4, %4, %12\n\tv_add_f32 %5, %5, %13\n\t"
            "v_add_f32 %6, %6, %14\n\tv_add_f32 %7, %7, %15\n\t"
            "s_mov_b64 exec, -1\n\ts_nop 0"
            : "+&v"(d[0]), "+&v"(d[1]), "+&v"(d[2]), "+&v"(d[3]), "+&v"(d[4]), "+&v"(d[5]), "+&v"(d[6]),
              "+&v"(d[7])
            : "v"(m[0]), "v"(m[1]), "v"(m[2]), "v"(m[3]), "v"(m[4]), "v"(m[5]), "v"(m[6]),
              "v"(m[7]), "i"(M));
}

// the lower (H = 0) or upper (H = 1) half of v in both halves of the wave
template <int H>
__device__ __forceinline__ float from_half(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[H]);
}

// -1/p from the hardware reciprocal and a Newton step in FMA: correctly
// rounded (checked against the division for every mantissa) while neither p
// nor 1/p comes near the ends of the exponent range; the kernel checks that
// on the results and factorises the panel again by divisions where it fails.
__device__ __forceinline__ bool rcp_in_range(float inv) {
    return ((__float_as_uint(inv) >> 23) & 0xffu) - 28u < 198u;
}

// Forward substitution of 4 NR vectors against a factorised 16 x 16 sub-block,
// an element per lane: lane (r, q) holds element r of vector 4 q' + k, k < NR.
//   SCALED: x_j *= dg_j, then x_r += x_j S[j][r], r > j (top strip)
//   else:   x_r += x_j S[j][r], r > j                   (left strip)
// S[j] is S[j][r] in lane r, dg lane r's dg_r.  A lane's element is scaled
// for its use at step j and, final by then, once more at the end.
template <bool SCALED, int NR>
__device__ __forceinline__ void solve16(float (&x)[NR], const float (&S)[16], float dg) {
#pragma clang fp contract(off)
    static_for<0, 15>([&](auto jc) {
        constexpr int j = jc.value;
        float u[NR];
#pragma unroll
        for (int k = 0; k < NR; ++k) u[k] = SCALED ? x[k] * dg : x[k];
#pragma unroll
        for (int k = 0; k < NR; ++k) u[k] = row_bcast<j>(u[k]) * S[j];
        add_in<above(j), NR>(x, u);
    });
    if (SCALED)
#pragma unroll
        for (int k = 0; k < NR; ++k) x[k] = x[k] * dg;
}

// a lane's 16 consecutive floats
__device__ __forceinline__ void read16(float (&S)[16], const float* p) {
#pragma unroll
    for (int g = 0; g < 16; g += 4) {
        const float4 v = *reinterpret_cast<const float4*>(p + g);
        S[g] = v.x;
        S[g + 1] = v.y;
        S[g + 2] = v.z;
        S[g + 3] = v.w;
    }
}

template <int B, int NT>
__global__ __launch_bounds__(NT) void lu_diag_kernel(float* __restrict__ A, int64_t lda,
                                                     int64_t off, int* __restrict__ status,
                                                     float* __restrict__ DT, int64_t ldt,
                                                     float* __restrict__ inv, int64_t inv_ts) {
#pragma clang fp contract(off)
    constexpr int LD = B + 4, NP = B / 16, NW = NT / 64, LS = 20;
    __shared__ __attribute__((aligned(16))) float Ds[B * LD];
    // the panel's left strip transposed (k-major); row 4 i + 2 e + h of each
    // block of 16 at 8 h + 4 e + i, the order in which a lane of the diagonal
    // update needs four of them
    __shared__ __attribute__((aligned(16))) float LT[16 * LD];
    __shared__ __attribute__((aligned(16))) float Sr[2 * 16 * LS];  // the sub-block transposed, by the panel's parity
    const int t = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    float* base = A + off * lda + off;
    constexpr int V = B * B / 4 / NT;
    static_assert(V >= 1 && V * NT * 4 == B * B, "block must split evenly over the threads");
    static_assert(NW >= 4, "waves 0, NW - 2 and NW - 1 have parts of their own");
    {
        float4 v[V];
#pragma unroll
        for (int i = 0; i < V; ++i) {
            const int e = t + i * NT, r = e / (B / 4), cc = (e % (B / 4)) * 4;
            v[i] = *reinterpret_cast<const float4*>(base + (int64_t)r * lda + cc);
        }
#pragma unroll
        for (int i = 0; i < V; ++i) {
            const int e = t + i * NT, r = e / (B / 4), cc = (e % (B / 4)) * 4;
            *reinterpret_cast<float4*>(&Ds[r * LD + cc]) = v[i];
        }
    }
    __syncthreads();

    // the rows and columns of panels lo..hi-1 (their parts outside earlier
    // panels') to the matrix and transposed to DT, by wave w of nw: a block of
    // 16 x 16 at a time, whose place is the same for the whole wave
    auto store = [&](int w, int nw, int lo, int hi) {
        const int lane = t & 63, y = lane >> 2, x = 4 * (lane & 3);
        float* ap = base + (int64_t)y * lda + x;
        float* dp = DT + (int64_t)y * ldt + x;
        for (int g = w; g < NP * NP; g += nw) {
            const int r0 = g / NP * 16, c0 = g % NP * 16, b = min(r0, c0) >> 4;
            if (b < lo || b >= hi) continue;
            const float4 v = *reinterpret_cast<const float4*>(&Ds[(r0 + y) * LD + c0 + x]);
            const float* q = &Ds[(c0 + x) * LD + r0 + y];
            const float4 d = {q[0], q[LD], q[2 * LD], q[3 * LD]};
            *reinterpret_cast<float4*>(ap + (int64_t)r0 * lda + c0) = v;
            *reinterpret_cast<float4*>(dp + (int64_t)r0 * ldt + c0) = d;
        }
    };
    // Panel p's part of the unit vectors' solves, for the top or the left strip's
    // recurrence: elements 0..15 of vectors 4 q + k of a 32 x 32 block in its
    // first half, elements 16..31 of those (from yu) and of vectors 16 + 4 q + k
    // (hi) in its second.
    float xu[4], yu[4];
    auto units = [&](int p, int lane, bool top, bool hi) {
        const int P0 = p * 16, r = lane & 15, q = lane >> 4;
        const bool odd = p & 1;
        float x[4], S[16];
#pragma unroll
        for (int k = 0; k < 4; ++k)
            x[k] = odd != hi ? (odd ? yu[k] : 0.0f) : (4 * q + k == r ? 1.0f : 0.0f);
        if (top) {
            read16(S, &Ds[(P0 + r) * LD + P0]);
            solve16<true, 4>(x, S, Ds[(P0 + r) * LD + P0 + r]);
        } else {
            read16(S, &Sr[(p & 1) * 16 * LS + r * LS]);
            solve16<false, 4>(x, S, 0.0f);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) xu[k] = x[k];
        // top: the inverse (S^-1 - C)^-1 of the top recurrence, stored
        // transposed, and its negated transpose, which is the inverse of the
        // sub-block's U
        const int row = (odd ? 16 : 0) + r, col = (hi ? 16 : 0) + 4 * q;
        float* o = inv + (top ? 0 : inv_ts) + (p >> 1) * 1024 + row + col * 32;
#pragma unroll
        for (int k = 0; k < 4; ++k) o[k * 32] = x[k];
        if (top)
            *reinterpret_cast<float4*>(inv + 2 * inv_ts + (p >> 1) * 1024 + row * 32 + col) =
                float4{-x[0], -x[1], -x[2], -x[3]};
    };
    bool bad = false;
#pragma unroll 1
    for (int p = 0; p <= NP; ++p) {
        const int P0 = p * 16;
        // opaque per panel: or every LDS address of the loop is formed before
        // it and held
        int lane = t & 63;
        asm volatile("" : "+v"(lane));
        const int r = lane & 15, q = lane >> 4;
        // ---- 1
        if (wave == 0 && p < NP) {
            const int c = r, e = q & 1, h = q >> 1;
            // lane (c, e, h): column P0 + c, rows 4 i + 2 e + h of the sub-block
            float z[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) z[i] = Ds[(P0 + 4 * i + 2 * e + h) * LD + P0 + c];
            if (p > 0) {
                const float* up = &Ds[(P0 - 16) * LD + P0 + c];
                const float* lp = &LT[P0 + 8 * h + 4 * e];
                float uv[16];
                float4 lv[16];
#pragma unroll
                for (int k = 0; k < 16; ++k) {
                    uv[k] = up[k * LD];
                    lv[k] = *reinterpret_cast<const float4*>(lp + k * LD);
                }
#pragma unroll
                for (int k = 0; k < 16; ++k) {
                    const float m0 = uv[k] * lv[k].x, m1 = uv[k] * lv[k].y;
                    const float m2 = uv[k] * lv[k].z, m3 = uv[k] * lv[k].w;
                    z[0] = z[0] + m0;
                    z[1] = z[1] + m1;
                    z[2] = z[2] + m2;
                    z[3] = z[3] + m3;
                }
            }
            // both e hold all rows 2 i + h
            float d[8], d0[8];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const auto w = __builtin_amdgcn_permlane16_swap(
                    __float_as_uint(z[i]), __float_as_uint(z[i]), false, false);
                d[2 * i] = __uint_as_float(w[0]);
                d[2 * i + 1] = __uint_as_float(w[1]);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) d0[i] = d[i];
            // V[j]: row j scaled by -1/pivot, in both halves; d keeps the columns
            // <= j of it, the multipliers and the pivot
            float V[16];
            const float piv0 = bcast(d[0], 0);
            float r0 = __builtin_amdgcn_rcpf(piv0);
            r0 = fmaf(fmaf(-piv0, r0, 1.0f), r0, r0);
            V[0] = from_half<0>(d[0]) * -r0;
            static_for<0, 15>([&](auto jc) {
                constexpr int j = jc.value, i1 = (j + 1) >> 1, h1 = (j + 1) & 1;
                float m[8];
#pragma unroll
                for (int i = i1; i < 8; ++i) m[i] = V[j] * row_bcast<j>(d[i]);
                add_in<above(j), 8 - i1>(d + i1, m + i1);
                const float piv = bcast(d[i1], h1 * 32 + j + 1);
                const float y = from_half<h1>(d[i1]);
                float rc = __builtin_amdgcn_rcpf(piv);
                rc = fmaf(fmaf(-piv, rc, 1.0f), rc, rc);
                V[j + 1] = y * -rc;
            });
            // -1/pivot of the lane's own column, where it has that row
            float dinv = 1.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (2 * i + h == c) dinv = d[i];
            {
                const float r1 = __builtin_amdgcn_rcpf(dinv);
                dinv = -fmaf(fmaf(-dinv, r1, 1.0f), r1, r1);
            }
            const bool fine = rcp_in_range(dinv);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float up = h ? V[2 * i + 1] : V[2 * i];
                d[i] = 2 * i + h == c ? dinv : 2 * i + h < c ? up : d[i];
            }
            if (__ballot(!fine)) {
                // a pivot near the ends of the exponent range (or zero): the
                // same steps with divisions, in LDS
#pragma unroll
                for (int i = 0; i < 8; ++i) Ds[(P0 + 2 * i + h) * LD + P0 + c] = d0[i];
                wave_lds_sync();
                for (int j = 0; j < 16; ++j) {
                    float* row = &Ds[(P0 + j) * LD + P0];
                    const float rinv = -1.0f / row[j];
                    const float s = c == j ? rinv : row[c] * rinv;
                    wave_lds_sync();
                    if (lane < 16 && c >= j) row[c] = s;
                    for (int rr = j + 1; rr < 16; ++rr) {
                        float* o = &Ds[(P0 + rr) * LD + P0];
                        const float u = s * o[j];
                        const float w = o[c] + u;
                        if (lane < 16 && c > j) o[c] = w;
                    }
                    wave_lds_sync();
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) d[i] = Ds[(P0 + 2 * i + h) * LD + P0 + c];
            }
            float* o = e ? &Sr[(p & 1) * 16 * LS + c * LS + h] : &Ds[(P0 + h) * LD + P0 + c];
            const int os = e ? 2 : 2 * LD;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                o[i * os] = d[i];
                if (2 * i + h == c) bad |= !__builtin_isfinite(d[i]);
            }
        } else if (wave > 0) {
            // panel p - 1's update of the w x w blocks of 16 without the first,
            // which is wave 0's: a row of 16 lanes per block, 4 x 4 per lane
            const int w = NP - p, nb = p > 0 ? w * w : 0;
            const int rcpw = 65536 / max(w, 1) + 1;
            for (int b0 = 4 * wave - 3; b0 < nb; b0 += 4 * (NW - 1)) {
                const bool in = b0 + q < nb;
                const int id = in ? b0 + q : b0;
                const int bi = (id * rcpw) >> 16, bj = id - bi * w;
                const int a = r >> 2, cc = P0 + 16 * bj + 4 * (r & 3);
                const int r0 = P0 + 16 * bi + 2 * (a & 1) + (a >> 1);  // rows r0 + 4 i
                const float* lp = &LT[P0 + 16 * bi + 4 * a];
                const float* up = &Ds[(P0 - 16) * LD + cc];
                float acc[4][4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float4 v = *reinterpret_cast<const float4*>(&Ds[(r0 + 4 * i) * LD + cc]);
                    acc[i][0] = v.x;
                    acc[i][1] = v.y;
                    acc[i][2] = v.z;
                    acc[i][3] = v.w;
                }
#pragma unroll 4
                for (int k = 0; k < 16; ++k) {
                    const float4 l = *reinterpret_cast<const float4*>(lp + k * LD);
                    const float4 u = *reinterpret_cast<const float4*>(up + k * LD);
                    const float lv[4] = {l.x, l.y, l.z, l.w}, uv[4] = {u.x, u.y, u.z, u.w};
                    float pr[4][4];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int b = 0; b < 4; ++b) pr[i][b] = uv[b] * lv[i];
#pragma unroll
                    for (int i = 0; i < 4; ++i)
#pragma unroll
                        for (int b = 0; b < 4; ++b) acc[i][b] = acc[i][b] + pr[i][b];
                }
                if (in)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        *reinterpret_cast<float4*>(&Ds[(r0 + 4 * i) * LD + cc]) =
                            float4{acc[i][0], acc[i][1], acc[i][2], acc[i][3]};
            }
            if (p > 0) {
                // waves NW - 1 and NW - 2 the low vectors, two others the high ones
                // (with four waves one takes both)
                if (wave < NW - 2)
                    for (int u = 0; u < 2; ++u) {
                        if (wave == (NW > 4 ? NW - 3 - u : 1)) units(p - 1, lane, u == 0, true);
                    }
                else
                    units(p - 1, lane, wave == NW - 1, false);
            }
            if ((p & 1) && wave >= NW - 2) {
                // elements 16..31 of the first 16 unit vectors
                const float* sp = wave == NW - 1
                                      ? &LT[P0 + (r & 1) * 8 + ((r >> 1) & 1) * 4 + (r >> 2)]
                                      : &Ds[(P0 - 16) * LD + P0 + r];
                float S[16];
#pragma unroll
                for (int j = 0; j < 16; ++j) S[j] = sp[j * LD];
#pragma unroll
                for (int k = 0; k < 4; ++k) yu[k] = 0.0f;
                static_for<0, 16>([&](auto jc) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const float u = row_bcast<jc.value>(xu[k]) * S[jc.value];
                        yu[k] = yu[k] + u;
                    }
                });
            }
            // what is final, where the updates leave time for it
            if (p >= NP / 2) {
                const int lo = min(2 * (p - NP / 2), NP - 1);
                // (of 16 waves, those that have neither a tile nor unit vectors)
                constexpr int W0 = NW > 8 ? 5 : 1, W1 = NW > 8 ? 12 : NW;
                if (wave >= W0 && wave < W1)
                    store(wave - W0, W1 - W0, lo, p == NP ? NP : min(lo + 2, p));
            }
        }
        if (p == NP) break;
        __syncthreads();
        // ---- 2
        const int R0 = P0 + 16, ng = NP - 1 - p;
        const float dg = Ds[(P0 + r) * LD + P0 + r];
        const float* scol = &Ds[(P0 + r) * LD + P0];
        const float* srow = &Sr[(p & 1) * 16 * LS + r * LS];
#pragma unroll 1
        for (int g = wave; g < 2 * ng; g += NW) {
            float x[4], S[16];
            if (g < ng) {
                float4* xp = reinterpret_cast<float4*>(&Ds[(P0 + r) * LD + R0 + 16 * g + 4 * q]);
                const float4 v = *xp;
                x[0] = v.x;
                x[1] = v.y;
                x[2] = v.z;
                x[3] = v.w;
                read16(S, scol);
                solve16<true, 4>(x, S, dg);
                *xp = float4{x[0], x[1], x[2], x[3]};
            } else {
                // register k: row 4 k + q of the group
                const int rr = R0 + 16 * (g - ng);
                float* xp = &Ds[(rr + q) * LD + P0 + r];
#pragma unroll
                for (int k = 0; k < 4; ++k) x[k] = xp[4 * k * LD];
                read16(S, srow);
                solve16<false, 4>(x, S, 0.0f);
#pragma unroll
                for (int k = 0; k < 4; ++k) xp[4 * k * LD] = x[k];
                *reinterpret_cast<float4*>(&LT[r * LD + rr + (q & 1) * 8 + (q >> 1) * 4]) =
                    float4{x[0], x[1], x[2], x[3]};
            }
        }
        __syncthreads();
    }
    if (bad && status) atomicMax(status, 1);
}

}  // namespace

hipError_t launch_lu_diag(float* A, int64_t lda, int64_t off, int B, int* status, float* DT,
                          int64_t ldt, float* inv, int64_t inv_ts, bool narrow, hipStream_t s) {
    // 16-byte row vectors
    if ((lda & 3) || (off & 3) || (ldt & 3) || (reinterpret_cast<uintptr_t>(A) & 15) ||
        (reinterpret_cast<uintptr_t>(DT) & 15) || !DT || !inv)
        return hipErrorInvalidValue;
#define HPL_LU(BB, NT)                                                                         \
    lu_diag_kernel<BB, NT><<<1, NT, 0, s>>>(A, lda, off, status, DT, ldt, inv, inv_ts)
    switch (B) {
        case 32: HPL_LU(32, 256); break;
        case 64:
            HPL_LU(64, 512);
            break;
        case 128:
            // 16 waves need a CU to themselves, which a large FP32 update beside
            // them does not leave: GEFA n = 32768 199.9 ms with 8 waves, 203.9
            // with 16, n = 16384 30.8 and 32.0; without one n = 2048 0.910 and
            // 0.860
            if (narrow) HPL_LU(128, 512);
            else HPL_LU(128, 1024);
            break;
        default: return hipErrorInvalidValue;
    }
#undef HPL_LU
    return hipGetLastError();
}
