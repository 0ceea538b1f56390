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
// One workgroup; the block lives in LDS and is processed in panels of 32
// pivot rows, three stages per panel:
//   A. wave 0 factorises the panel's 32 x 32 diagonal sub-block.  The other
//      waves apply the previous panel's rank-32 update to the blocks that
//      this panel's stage C does not need, and at the last panel store what
//      is finished.
//   B. every column right of the sub-block (top strip) and every row below it
//      (left strip) is solved against the sub-block, 32 vectors per wave, and
//      one further wave of each kind solves for the 32 unit vectors: those
//      are the sub-block's inverses.
//   C. the next diagonal sub-block alone receives this panel's update.
// So the chain from pivot to pivot holds A, one strip solve and one 32 x 32
// update per panel, not the whole trailing update.
//
// Bound: instruction latency of stage A's single wave (a pivot step is about
// 45 instructions, 320 cycles) and of the 32-step strip solves (180 cycles a
// step).  In A and B a lane holds 16 values of one vector -- rows (or
// columns) of one parity, the two halves of the wave holding the two
// parities -- so a step's updates take half the instructions of one lane per
// vector.  A's multipliers are broadcast within each half by ds_swizzle right
// after the row's update, one step ahead of their use; the next pivot's row
// goes first and its reciprocal's chain is issued between the other rows.
// B = 128 alone on the device: 39.6 us with the inverses and DT, against
// 62.2 us for the former one-stage-at-a-time kernel and a further launch of 8
// us for those (B = 64: 21.3 against 26.1 + 8; B = 32: 11.0 against 9.2 + 7);
// GEFA + GESL at n = 2048, B = 128: 2.36 -> 1.91 ms.
// At most 128 VGPRs and 91 KiB of LDS: the workgroup fits into what one of
// the two workgroups of the FP32 trailing update on a CU leaves, whichever of
// the two ends first (with 109 KiB, a second buffer of the left strip, only
// after the second one: 4% on n = 32768).
// Blocks up to 128 are handled here; larger diagonal blocks are factorised by
// the host schedule as a 2 x 2 recursion on top of this kernel.
#include "common.hpp"
#include "kernels.hpp"

#include <type_traits>

namespace {

__device__ __forceinline__ float bcast(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// b where the mask has the lane, else a
__device__ __forceinline__ float pick(unsigned long long mask, float a, float b) {
    float r;
    asm("v_cndmask_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "s"(mask));
    return r;
}

constexpr unsigned long long kLowHalf = 0xffffffffull, kHighHalf = kLowHalf << 32;

// d[i] += m[i], i < n <= 4, in the lanes of the mask: one change of the exec
// mask instead of a select per value (every lane of the wave is active here)
__device__ __forceinline__ void add_in(unsigned long long mask, int n, float* d, const float* m) {
    if (n == 4)
        asm("s_mov_b64 exec, %8\n\tv_add_f32 %0, %0, %4\n\tv_add_f32 %1, %1, %5\n\t"
            "v_add_f32 %2, %2, %6\n\tv_add_f32 %3, %3, %7\n\ts_mov_b64 exec, -1"
            : "+v"(d[0]), "+v"(d[1]), "+v"(d[2]), "+v"(d[3])
            : "v"(m[0]), "v"(m[1]), "v"(m[2]), "v"(m[3]), "s"(mask));
    else if (n == 3)
        asm("s_mov_b64 exec, %6\n\tv_add_f32 %0, %0, %3\n\tv_add_f32 %1, %1, %4\n\t"
            "v_add_f32 %2, %2, %5\n\ts_mov_b64 exec, -1"
            : "+v"(d[0]), "+v"(d[1]), "+v"(d[2])
            : "v"(m[0]), "v"(m[1]), "v"(m[2]), "s"(mask));
    else if (n == 2)
        asm("s_mov_b64 exec, %4\n\tv_add_f32 %0, %0, %2\n\tv_add_f32 %1, %1, %3\n\t"
            "s_mov_b64 exec, -1"
            : "+v"(d[0]), "+v"(d[1])
            : "v"(m[0]), "v"(m[1]), "s"(mask));
    else
        asm("s_mov_b64 exec, %2\n\tv_add_f32 %0, %0, %1\n\ts_mov_b64 exec, -1"
            : "+v"(d[0])
            : "v"(m[0]), "s"(mask));
}

// lane J of each half of the wave to all lanes of that half
template <int J>
__device__ __forceinline__ float half_bcast(float v) {
    return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), J << 5));
}

// the lower (H = 0) or upper (H = 1) half of v in both halves of the wave
template <int H>
__device__ __forceinline__ float from_half(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[H]);
}

template <int J, typename F>
__device__ __forceinline__ void static_for32(F&& f) {
    if constexpr (J < 32) {
        f(std::integral_constant<int, J>{});
        static_for32<J + 1>(f);
    }
}

// -1/p from the hardware reciprocal and two Newton steps in FMA: correctly
// rounded (checked against the division for every mantissa) while neither p
// nor 1/p comes near the ends of the exponent range; the kernel checks that
// on the results and factorises the panel again by divisions where it fails.
__device__ __forceinline__ bool rcp_in_range(float inv) {
    return ((__float_as_uint(inv) >> 23) & 0xffu) - 28u < 198u;
}

// Forward substitution of one vector per half-lane pair against the
// factorised sub-block: lane (c, h) holds x[i] = element 2 i + h of vector c.
//   SCALED: x_j *= dg_j, then x_r += x_j S[j][r], r > j (top strip)
//   else:   x_r += x_j S[j][r], r > j                   (left strip)
// with S[j][r] at S[32 j + 16 (r % 2) + r / 2]: a step's coefficients are
// 16-byte LDS broadcasts, read two steps ahead.
template <bool SCALED>
__device__ __forceinline__ void solve32(float (&x)[16], const float* S, float dgl, int h) {
#pragma clang fp contract(off)
    float dg[SCALED ? 32 : 1];
    if constexpr (SCALED) {
#pragma unroll
        for (int j = 0; j < 32; ++j) dg[j] = bcast(dgl, j);
    }
    const float* Sh = S + h * 16;
    float4 nx[2][4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        nx[0][g] = *reinterpret_cast<const float4*>(Sh + 4 * g);
        nx[1][g] = *reinterpret_cast<const float4*>(Sh + 32 + 4 * g);
    }
    static_for32<0>([&](auto jc) {
        constexpr int j = jc.value, i0 = j >> 1, hj = j & 1;
        float s4[16];
#pragma unroll
        for (int g = (i0 + hj) / 4; g < 4; ++g) {
            float4& q = nx[hj][g];
            // whole 16-byte reads, also where a step needs part of one
            asm volatile("" : "+v"(q.x), "+v"(q.y), "+v"(q.z), "+v"(q.w));
            s4[4 * g] = q.x;
            s4[4 * g + 1] = q.y;
            s4[4 * g + 2] = q.z;
            s4[4 * g + 3] = q.w;
        }
        if constexpr (j < 30) {
#pragma unroll
            for (int g = (j + 3) / 8; g < 4; ++g)
                nx[hj][g] = *reinterpret_cast<const float4*>(Sh + (j + 2) * 32 + 4 * g);
        }
        float s = x[i0];
        if constexpr (SCALED) s = s * dg[j];
        const float v = from_half<hj>(s);
        if constexpr (SCALED) x[i0] = pick(hj ? kHighHalf : kLowHalf, x[i0], s);
        if constexpr (hj == 0) {
            const float u = v * s4[i0];
            const float w = x[i0] + u;
            x[i0] = pick(kHighHalf, x[i0], w);
        }
#pragma unroll
        for (int i = i0 + 1; i < 16; ++i) s4[i] = v * s4[i];
#pragma unroll
        for (int i = i0 + 1; i < 16; ++i) x[i] = x[i] + s4[i];
        __builtin_amdgcn_sched_barrier(0);
    });
}

template <int B, int NT>
__global__ __launch_bounds__(NT) void lu_diag_kernel(float* __restrict__ A, int64_t lda,
                                                     int64_t off, int* __restrict__ status,
                                                     float* __restrict__ DT, int64_t ldt,
                                                     float* __restrict__ inv, int64_t inv_ts) {
#pragma clang fp contract(off)
    constexpr int LD = B + 4, NP = B / 32, NW = NT / 64;
    __shared__ __attribute__((aligned(16))) float Ds[B * LD];
    // the panel's left strip transposed (k-major)
    __shared__ __attribute__((aligned(16))) float LT[B > 32 ? 32 * LD : 4];
    // the factorised sub-block by columns and by rows, each column's (row's)
    // even elements before its odd ones
    __shared__ __attribute__((aligned(16))) float Sc[1024], Sr[1024];
    const int t = threadIdx.x;
    const int wave = t >> 6;
    int lane = t & 63, c = lane & 31, h = lane >> 5;
    float* base = A + off * lda + off;
    constexpr int V = B * B / 4 / NT;
    static_assert(V >= 1 && V * NT * 4 == B * B, "block must split evenly over the threads");
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

    // rank-32 update of the 4 x 4 register tile of each lane in the 32 x 32
    // block (bi, bj) by panel q
    auto tile32 = [&](int q, int bi, int bj) {
        const int rr = bi * 32 + (lane >> 3) * 4, cc = bj * 32 + (lane & 7) * 4;
        float acc[4][4];
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            const float4 v = *reinterpret_cast<const float4*>(&Ds[(rr + a) * LD + cc]);
            acc[a][0] = v.x;
            acc[a][1] = v.y;
            acc[a][2] = v.z;
            acc[a][3] = v.w;
        }
        const float* lt = &LT[rr];
        const float* tp = &Ds[q * 32 * LD + cc];
#pragma unroll 4
        for (int k = 0; k < 32; ++k) {
            const float4 l = *reinterpret_cast<const float4*>(lt + k * LD);
            const float4 u = *reinterpret_cast<const float4*>(tp + k * LD);
            const float lv[4] = {l.x, l.y, l.z, l.w}, uv[4] = {u.x, u.y, u.z, u.w};
            float pr[4][4];
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) pr[a][b] = uv[b] * lv[a];
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) acc[a][b] = acc[a][b] + pr[a][b];
        }
#pragma unroll
        for (int a = 0; a < 4; ++a)
            *reinterpret_cast<float4*>(&Ds[(rr + a) * LD + cc]) =
                float4{acc[a][0], acc[a][1], acc[a][2], acc[a][3]};
    };
    // the same for the 16 x 16 quarter qt of block (b, b), 2 x 2 per lane
    auto tile16 = [&](int q, int b, int qt) {
        const int rr = b * 32 + (qt >> 1) * 16 + (lane >> 3) * 2;
        const int cc = b * 32 + (qt & 1) * 16 + (lane & 7) * 2;
        float acc[2][2];
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            acc[a][0] = Ds[(rr + a) * LD + cc];
            acc[a][1] = Ds[(rr + a) * LD + cc + 1];
        }
        const float* lt = &LT[rr];
        const float* tp = &Ds[q * 32 * LD + cc];
        // the next four operand pairs are read while four are multiplied
        float2 l[4], u[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            l[k] = *reinterpret_cast<const float2*>(lt + k * LD);
            u[k] = *reinterpret_cast<const float2*>(tp + k * LD);
        }
#pragma unroll 1
        for (int kb = 4; kb <= 32; kb += 4) {
            float2 ln[4], un[4];
            const int kn = kb < 32 ? kb : 28;  // the last turn reads again what it has
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                ln[k] = *reinterpret_cast<const float2*>(lt + (kn + k) * LD);
                un[k] = *reinterpret_cast<const float2*>(tp + (kn + k) * LD);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float p0 = u[k].x * l[k].x, p1 = u[k].y * l[k].x;
                const float p2 = u[k].x * l[k].y, p3 = u[k].y * l[k].y;
                acc[0][0] = acc[0][0] + p0;
                acc[0][1] = acc[0][1] + p1;
                acc[1][0] = acc[1][0] + p2;
                acc[1][1] = acc[1][1] + p3;
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                l[k] = ln[k];
                u[k] = un[k];
            }
        }
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            Ds[(rr + a) * LD + cc] = acc[a][0];
            Ds[(rr + a) * LD + cc + 1] = acc[a][1];
        }
    };
    // the elements of the last 32 x 32 block, or all others, to the matrix and
    // transposed to DT: 8 rows x 8 float4 columns per wave, so that a wave's
    // stores fill 128-byte lines and its LDS reads by column meet few conflicts
    auto store = [&](int s, int ns, bool last) {
        constexpr int G = B / 8, GC = B / 32;
        for (int g = s >> 6; g < G * GC; g += ns >> 6) {
            const int r = (g / GC) * 8 + (s & 7), cc = (g % GC) * 32 + ((s >> 3) & 7) * 4;
            if (last != (r >= B - 32 && cc >= B - 32)) continue;
            const int r2 = (g / GC) * 8 + ((s >> 3) & 7), c2 = (g % GC) * 32 + (s & 7) * 4;
            *reinterpret_cast<float4*>(base + (int64_t)r2 * lda + c2) =
                *reinterpret_cast<const float4*>(&Ds[r2 * LD + c2]);
            *reinterpret_cast<float4*>(DT + (int64_t)r * ldt + cc) =
                float4{Ds[cc * LD + r], Ds[(cc + 1) * LD + r], Ds[(cc + 2) * LD + r],
                       Ds[(cc + 3) * LD + r]};
        }
    };
    bool bad = false;
#pragma unroll 1
    for (int p = 0; p < NP; ++p) {
        const int P0 = p * 32;
        // opaque per panel: or every LDS address of the loop is formed before
        // it and held (100 registers)
        lane = t & 63;
        asm volatile("" : "+v"(lane));
        c = lane & 31;
        h = lane >> 5;
        // ---- A: lane (c, h) holds rows 2 i + h of column P0 + c
        if (wave == 0) {
            float d[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) d[i] = Ds[(P0 + 2 * i + h) * LD + P0 + c];
            // lanes (both halves) whose column is above j, shifted along: kept
            // out of the compiler's sight, or it hoists and spills 32 masks
            unsigned long long gt = 0xfffffffefffffffeull;
            asm volatile("" : "+s"(gt));
            float m[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) m[i] = half_bcast<0>(d[i]);
            // row j scaled by -1/pivot, the pivot itself replaced by -1/pivot
            const float piv0 = bcast(d[0], 0);
            float r0 = __builtin_amdgcn_rcpf(piv0);
            r0 = fmaf(fmaf(-piv0, r0, 1.0f), r0, r0);
            r0 = fmaf(fmaf(-piv0, r0, 1.0f), r0, r0);
            float sc = pick(1ull, d[0], 1.0f) * -r0;
            static_for32<0>([&](auto jc) {
                constexpr int j = jc.value, i0 = j >> 1, hj = j & 1;
                constexpr int j1 = (j + 1) & 31, i1 = j1 >> 1, h1 = j1 & 1;
                const unsigned long long ge = gt | (1ull << j) | (1ull << (j + 32));
                // row j scaled, in both halves
                const float v = from_half<hj>(sc);
                if constexpr (j < 31) {
                    // the next pivot's row first; its reciprocal's chain goes
                    // between the other rows' updates
                    float u = v * m[i1], w = d[i1] + u;
                    d[i0] = pick(ge & (hj ? kHighHalf : kLowHalf), d[i0], sc);
                    d[i1] = pick(hj == 0 ? gt & kHighHalf : gt, d[i1], w);
                    const float piv = bcast(d[i1], h1 * 32 + j1);
                    if constexpr (h1 == 0) m[i1] = half_bcast<j1>(d[i1]);
                    float r = __builtin_amdgcn_rcpf(piv), e = 0.0f, x1 = 0.0f;
                    auto link = [&](int n) {
                        if (n == 0) x1 = pick(1ull << (j1 + 32 * h1), d[i1], 1.0f);
                        if (n == 1) e = fmaf(-piv, r, 1.0f);
                        if (n == 2) r = fmaf(e, r, r);
                        if (n == 3) e = fmaf(-piv, r, 1.0f);
                        if (n == 4) r = fmaf(e, r, r);
                        if (n == 5) sc = x1 * -r;
                        __builtin_amdgcn_sched_barrier(0);
                    };
                    __builtin_amdgcn_sched_barrier(0);
                    // four rows at a time, operation by operation: a result
                    // is not ready for the next instruction
                    constexpr int NG = (15 - i1 + 3) / 4;
#pragma unroll
                    for (int g = 0; g < NG; ++g) {
                        const int ia = i1 + 1 + 4 * g, ib = ia + 4 < 16 ? ia + 4 : 16;
                        asm volatile("" : "+v"(m[ib - 1]));  // one wait for the group's values
#pragma unroll
                        for (int i = ia; i < ib; ++i) m[i] = v * m[i];
                        link(2 * g);
                        add_in(gt, ib - ia, d + ia, m + ia);
                        link(2 * g + 1);
#pragma unroll
                        for (int i = ia; i < ib; ++i) m[i] = half_bcast<j1>(d[i]);
                        __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int n = 2 * NG; n < 6; ++n) link(n);
                } else {
                    d[i0] = pick(ge & (hj ? kHighHalf : kLowHalf), d[i0], sc);
                }
                gt = (gt & 0x7fffffff7fffffffull) << 1;
            });
            bool fine = true;
#pragma unroll
            for (int i = 0; i < 16; ++i)
                if (2 * i + h == c) fine = rcp_in_range(d[i]);
            if (__ballot(!fine)) {
                // a pivot near the ends of the exponent range (or zero): the
                // same steps with divisions, on the panel as it still lies in LDS
                for (int j = 0; j < 32; ++j) {
                    float* row = &Ds[(P0 + j) * LD + P0];
                    const float rinv = -1.0f / row[j];
                    const float s = c == j ? rinv : row[c] * rinv;
                    wave_lds_sync();
                    if (lane < 32 && c >= j) row[c] = s;
                    for (int r = j + 1; r < 32; ++r) {
                        float* q = &Ds[(P0 + r) * LD + P0];
                        const float u = s * q[j];
                        const float w = q[c] + u;
                        if (lane < 32 && c > j) q[c] = w;
                    }
                    wave_lds_sync();
                }
#pragma unroll
                for (int i = 0; i < 16; ++i) d[i] = Ds[(P0 + 2 * i + h) * LD + P0 + c];
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int r = 2 * i + h;
                Ds[(P0 + r) * LD + P0 + c] = d[i];
                Sr[r * 32 + (c & 1) * 16 + (c >> 1)] = d[i];
                if (r == c) bad |= !__builtin_isfinite(d[i]);
            }
#pragma unroll
            for (int i = 0; i < 16; i += 4)
                *reinterpret_cast<float4*>(&Sc[c * 32 + h * 16 + i]) =
                    float4{d[i], d[i + 1], d[i + 2], d[i + 3]};
        } else if (NP == 4 && (p == 1 || p == 2)) {
            // panel p - 1's update of blocks p..3 x p..3 without (p, p), which is done
            const int w = 4 - p;
            for (int x = wave; x < w * w; x += NW - 1) tile32(p - 1, p + x / w, p + x % w);
        }
        if (NP > 1 && p == NP - 1 && wave > 0) store(t - 64, NT - 64, false);
        __syncthreads();
        // ---- B: wave g the top group g, wave ng the unit vectors, then the same
        // of the left strip
        const int R0 = P0 + 32;
        const int ng = NP - 1 - p;
#pragma unroll 1
        for (int g = wave; g < 2 * (ng + 1); g += NW) {
            float x[16];
            if (g <= ng) {
                const bool unit = g == ng;
                const int cc = unit ? P0 + c : R0 + g * 32 + c;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const float v = Ds[(P0 + 2 * i + h) * LD + cc];
                    x[i] = unit ? (2 * i + h == c ? 1.0f : 0.0f) : v;
                }
                solve32<true>(x, Sc, Sc[c * 32 + (c & 1) * 16 + (c >> 1)], h);
                if (unit) {
                    // the inverse (S^-1 - C)^-1 of the top recurrence, stored
                    // transposed, and its negated transpose, which is the
                    // inverse of the sub-block's U
                    float* o = inv + p * 1024;
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        o[c * 32 + 2 * i + h] = x[i];
                        o[2 * inv_ts + (2 * i + h) * 32 + c] = -x[i];
                    }
                } else {
#pragma unroll
                    for (int i = 0; i < 16; ++i) Ds[(P0 + 2 * i + h) * LD + cc] = x[i];
                }
            } else {
                const bool unit = g == 2 * ng + 1;
                const int rr = unit ? P0 + c : R0 + (g - ng - 1) * 32 + c;
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const float v = Ds[rr * LD + P0 + 2 * i + h];
                    x[i] = unit ? (2 * i + h == c ? 1.0f : 0.0f) : v;
                }
                solve32<false>(x, Sr, 0.0f, h);
                if (unit) {
                    float* o = inv + inv_ts + p * 1024 + c * 32 + h;
#pragma unroll
                    for (int i = 0; i < 16; ++i) o[2 * i] = x[i];
                } else {
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        Ds[rr * LD + P0 + 2 * i + h] = x[i];
                        LT[(2 * i + h) * LD + rr] = x[i];
                    }
                }
            }
        }
        if (p + 1 == NP) {
            if (wave >= 2) store(t - 128, NT - 128, true);
            break;
        }
        __syncthreads();
        // ---- C: (1, 1), (2, 2), (3, 3)
        if (wave < 4) tile16(p, p + 1, wave);
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
            if (narrow) HPL_LU(64, 256);
            else HPL_LU(64, 512);
            break;
        case 128:
            if (narrow) HPL_LU(128, 256);
            else HPL_LU(128, 512);
            break;
        default: return hipErrorInvalidValue;
    }
#undef HPL_LU
    return hipGetLastError();
}
