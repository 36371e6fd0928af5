// int8 weight-only GEMM on MFMA for gfx950: the q8 linear beyond the few rows
// that the GEMV (qlinear.hpp) serves.
//
// Arithmetic spec: q8_matvec (crates/tang-infer/src/quantize.rs:227-254) per
// activation row.
#pragma once

#include "qlinear.hpp"

namespace th {

// Four int8 values of one word as two bf16 pairs (exact: |w| <= 128).
__device__ __forceinline__ void i8x4_to_bf16(uint32_t w, uint32_t& p0, uint32_t& p1) {
    const uint32_t f0 = __float_as_uint((float)(int8_t)w), f1 = __float_as_uint((float)(int8_t)(w >> 8));
    const uint32_t f2 = __float_as_uint((float)(int8_t)(w >> 16)), f3 = __float_as_uint((float)(int8_t)(w >> 24));
    p0 = __builtin_amdgcn_perm(f1, f0, 0x07060302u);
    p1 = __builtin_amdgcn_perm(f3, f2, 0x07060302u);
}

// Eight f32 values times 2^EXP as three bf16 parts, x = p[0] + p[1] + p[2]
// exactly: each part takes the next eight significant bits by truncation, and
// both differences are exact in f32.  Where the last part lies below bf16's
// subnormals (an |x| under 2^-110, unscaled) the half of its word that is lost
// goes to the low half of `lost`.  EXP = SPLIT_EXP leaves nothing of the
// smallest subnormal out, but takes eight multiplications that a GEMM's step
// feels (matmul m 509, k 2048, n 5632: 66 -> 76 us).  Non-finite values, and
// those from 2^(128 - EXP) on, give NaN.
constexpr int SPLIT_EXP = 16;
template <int EXP>
__device__ __forceinline__ void split3_bf16(const uint4& a, const uint4& b, uint4 (&p)[3], uint32_t& lost) {
    const uint32_t x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    uint32_t v[8], m[8], l[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        v[i] = EXP ? __float_as_uint(__uint_as_float(x[i]) * (float)(1 << EXP)) : x[i];
        const float r1 = __uint_as_float(v[i]) - __uint_as_float(v[i] & 0xFFFF0000u);
        m[i] = __float_as_uint(r1);
        l[i] = __float_as_uint(r1 - __uint_as_float(m[i] & 0xFFFF0000u));
    }
#pragma unroll
    for (int i = 0; i < 8; i += 2) lost |= l[i] | l[i + 1];
    auto pk = [](const uint32_t (&h)[8]) {  // the high halves, in element order
        return make_uint4(__builtin_amdgcn_perm(h[1], h[0], 0x07060302u), __builtin_amdgcn_perm(h[3], h[2], 0x07060302u),
                          __builtin_amdgcn_perm(h[5], h[4], 0x07060302u), __builtin_amdgcn_perm(h[7], h[6], 0x07060302u));
    };
    p[0] = pk(v);
    p[1] = pk(m);
    p[2] = pk(l);
}

// Workgroup: 4 waves along the weight rows, RT 16-row tiles each, times CB
// blocks of 16 activation rows; K in steps of KG 64-wide chunks, the
// activations double-buffered in LDS (one barrier a step), each wave's
// weights straight from memory to its registers.  v_mfma_f32_16x16x32_bf16
// with A = activations (bf16 rows as they are, f32 rows as three bf16 parts:
// every product exact), B = weights (int8 is exact in bf16).  A tile's lane
// (q, r) holds k 16q..16q+15 of its chunk, so lanes 0-31 hold the first
// 32-group and lanes 32-63 the second; v_permlane32_swap hands each half's
// upper eight to the other, after which one MFMA covers exactly one 32-group,
// its k octets in the order 0, 2, 1, 3.  With a scale per group each MFMA
// starts from zero and its D is weighted with one FMA by the lane's scale
// (the lane's D column is one weight row); with a scale per row the MFMAs
// accumulate and the scale comes at the end.  A step sums up by itself before
// it joins the accumulators: short chains of f32 additions, as the GEMV's.  A
// workgroup that met f32 values with vanishing parts (split3_bf16) makes a
// second, scaled pass; finding them costs 3 to 6% (m = 100: 48 -> 51 us per-row
// scales, 52 -> 56 per-group).
//
// Bound by the weight stream up to about 32 rows, then by the conversions and
// scale FMAs next to the MFMAs: 11008 x 4096, per-group scales, bf16 rows:
// m = 32 184 -> 20 us (2.6 TB/s), m = 100 570 -> 34 us (262 TFLOP/s).
// Three waves per SIMD and 64-row blocks: 128-row ones leave one (m = 100: 80
// us).  Plain weight loads: each block of 64 rows reads the weights again, and
// non-temporal ones measured 43 against 37 us there.
template <int RT, int CB, int KG, bool XF32, bool VEC, bool PER_ROW, int WPE = 3>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WPE))) void q8_gemm_kernel(const uint4* __restrict__ wt, const float* __restrict__ sc,
                                                      const void* __restrict__ xin, float* __restrict__ y, int M,
                                                      int N, int K, int Kp, int ldx, int ldy, size_t split_stride,
                                                      int ch_per_split) {
    constexpr int PARTS = XF32 ? 3 : 1;
    constexpr int OCT = 8 * KG;               // 8-value octets of a row per step
    constexpr int LD = 17;                    // octet stride in 16-byte units (16 rows + 1: spreads the banks)
    constexpr int PLANE = CB * OCT * LD;      // one part of a step
    constexpr int NOCT = CB * 16 * OCT;       // octets staged per step
    constexpr int PT = (NOCT + 255) / 256;    // octets per thread
    __shared__ uint4 xt[2][PARTS * PLANE];
    int bx = blockIdx.x, by = blockIdx.y, split = blockIdx.z;
    gemm_xcd_tile(bx, by, split);
    uint32_t lost = 0;
    auto pass = [&](auto ex) {  // f32 rows times 2^ex
        constexpr int EXP = decltype(ex)::value;
        int tid = threadIdx.x;
        if constexpr (XF32) asm volatile("" : "+v"(tid));  // a second pass forms its places again: none kept through the first
        const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int q = lane >> 4, r = lane & 15;
        const int NCH = Kp >> 6, NT = (N + 15) >> 4, GPR = Kp >> 5;
        const int c0 = split * ch_per_split, c1 = min(NCH, c0 + ch_per_split);
        const int m0 = by * CB * 16, mrows = min(CB * 16, M - m0);
        const int tile0 = (bx * 4 + wave) * RT;
        const int octq = ((q & 1) << 1) | (q >> 1);  // octet of a 32-group that this lane multiplies

        // Activation octets of a step: thread -> (row, octet), eight (or sixteen)
        // consecutive threads per row.  Rows past the block re-read its last row
        // (never stored); octets past K are zeroed when stored.
        u32x4_t xa[PT], xb[XF32 ? PT : 1];  // native vectors: arrays of uint4 structs go to scratch
        auto load_x = [&](int c) {
#pragma unroll
            for (int i = 0; i < PT; i++) {
                const int idx = min(tid + 256 * i, NOCT - 1), row = min(idx / OCT, mrows - 1), o = idx % OCT;
                uint4 a, b;
                load_x8<XF32, VEC>(xin, m0 + row, ldx, K, c * 64 + o * 8, a, b);
                xa[i] = __builtin_bit_cast(u32x4_t, a);
                if constexpr (XF32) xb[i] = __builtin_bit_cast(u32x4_t, b);
            }
        };
        auto store_x = [&](uint4* t, int c) {
#pragma unroll
            for (int i = 0; i < PT; i++) {
                const int idx = tid + 256 * i, row = idx / OCT, o = idx % OCT;
                if (NOCT % 256 != 0 && idx >= NOCT) break;
                const uint4 z = make_uint4(0, 0, 0, 0);
                const bool in = c * 64 + o * 8 < K;
                uint4* dst = t + ((row >> 4) * OCT + o) * LD + (row & 15);
                if constexpr (XF32) {
                    uint4 p[3];
                    split3_bf16<EXP>(in ? __builtin_bit_cast(uint4, xa[i]) : z, in ? __builtin_bit_cast(uint4, xb[i]) : z, p, lost);
#pragma unroll
                    for (int e = 0; e < 3; e++) dst[e * PLANE] = p[e];
                } else {
                    *dst = in ? __builtin_bit_cast(uint4, xa[i]) : z;
                }
            }
        };
        u32x4_t wcur[RT][KG], wnxt[RT][KG];
        float scur[RT][KG][2], snxt[RT][KG][2];
        auto load_w = [&](int c, u32x4_t (&w)[RT][KG], float (&s)[RT][KG][2]) {
#pragma unroll
            for (int a = 0; a < RT; a++) {
                const int t = min(tile0 + a, NT - 1);
#pragma unroll
                for (int k = 0; k < KG; k++) {
                    const int ck = min(c + k, NCH - 1);
                    w[a][k] = *(const u32x4_t*)(wt + ((size_t)t * NCH + ck) * 64 + lane);
                    if constexpr (!PER_ROW) {
                        const float2 v = *(const float2*)(sc + (size_t)(t * 16 + r) * GPR + 2 * ck);
                        s[a][k][0] = v.x;
                        s[a][k][1] = v.y;
                    }
                }
            }
        };
        float4_t acc[RT][CB];
#pragma unroll
        for (int a = 0; a < RT; a++)
#pragma unroll
            for (int b = 0; b < CB; b++) acc[a][b] = (float4_t){0.0f, 0.0f, 0.0f, 0.0f};
        load_x(c0);
        load_w(c0, wcur, scur);
        store_x(xt[0], c0);
        __syncthreads();
        int buf = 0;
        for (int c = c0; c < c1; c += KG) {
            const uint4* t = xt[buf];
            const bool more = c + KG < c1;
            if (more) {
                load_x(c + KG);
                load_w(c + KG, wnxt, snxt);
            }
            bf16x8_t bw[RT][KG][2];
#pragma unroll
            for (int a = 0; a < RT; a++)
#pragma unroll
                for (int k = 0; k < KG; k++) {
                    // the last step's missing chunk (its activations are zeros
                    // past K) multiplies nothing
                    const u32x4_t w = c + k < c1 ? wcur[a][k] : (u32x4_t){0, 0, 0, 0};
                    const auto s0 = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false);
                    const auto s1 = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
#pragma unroll
                    for (int g = 0; g < 2; g++) {
                        uint4 f;
                        i8x4_to_bf16(s0[g], f.x, f.y);
                        i8x4_to_bf16(s1[g], f.z, f.w);
                        bw[a][k][g] = __builtin_bit_cast(bf16x8_t, f);
                    }
                }
#pragma unroll
            for (int b = 0; b < CB; b++) {
                bf16x8_t af[KG][2][PARTS];
#pragma unroll
                for (int k = 0; k < KG; k++)
#pragma unroll
                    for (int g = 0; g < 2; g++)
#pragma unroll
                        for (int p = 0; p < PARTS; p++)
                            af[k][g][p] = __builtin_bit_cast(bf16x8_t, t[p * PLANE + (b * OCT + k * 8 + g * 4 + octq) * LD + r]);
#pragma unroll
                for (int a = 0; a < RT; a++) {
                    float4_t v = {0.0f, 0.0f, 0.0f, 0.0f};  // this step's sum: joins acc once
#pragma unroll
                    for (int k = 0; k < KG; k++)
#pragma unroll
                        for (int g = 0; g < 2; g++) {
                            float4_t d = PER_ROW ? v : (float4_t){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                            for (int p = PARTS - 1; p >= 0; p--)
                                d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[k][g][p], bw[a][k][g], d, 0, 0, 0);
                            if constexpr (PER_ROW) {
                                v = d;
                            } else {
#pragma unroll
                                for (int e = 0; e < 4; e++) v[e] = __builtin_fmaf(scur[a][k][g], d[e], v[e]);
                            }
                        }
                    acc[a][b] += v;
                }
                if constexpr (!PER_ROW) {
                    // The next block's MFMAs take the weights from here on: left
                    // alone the compiler runs every block's MFMAs first, and their
                    // results (16 registers a tile and step) spill or cost the
                    // SIMD its second and third wave.
#pragma unroll
                    for (int a = 0; a < RT; a++)
#pragma unroll
                        for (int k = 0; k < KG; k++)
                            asm volatile("" : "+v"(acc[a][b]), "+v"(bw[a][k][0]), "+v"(bw[a][k][1]));
                }
            }
#pragma unroll
            for (int a = 0; a < RT; a++)
#pragma unroll
                for (int b = 0; b < CB; b++) mfma_pin(acc[a][b]);
            buf ^= 1;  // last read in the step before, ordered by that step's barrier
            if (more) store_x(xt[buf], c + KG);
            __syncthreads();
#pragma unroll
            for (int a = 0; a < RT; a++)
#pragma unroll
                for (int k = 0; k < KG; k++) {
                    wcur[a][k] = wnxt[a][k];
                    scur[a][k][0] = snxt[a][k][0];
                    scur[a][k][1] = snxt[a][k][1];
                }
        }
        float* yb = y + (size_t)split * split_stride;
#pragma unroll
        for (int a = 0; a < RT; a++) {
            const int n = (tile0 + a) * 16 + r;
            if (n >= N) continue;
            const float s = PER_ROW ? sc[n] : 1.0f;
#pragma unroll
            for (int b = 0; b < CB; b++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int m = b * 16 + 4 * q + e;
                    const float v = EXP ? __builtin_amdgcn_ldexpf(acc[a][b][e], -EXP) : acc[a][b][e];
                    if (m < mrows && (!EXP || fabsf(v) <= 3.402823466e38f)) yb[(size_t)(m0 + m) * ldy + n] = v * s;
                }
        }
    };
    pass(std::integral_constant<int, 0>{});
    if constexpr (XF32) {
        // Rows with vanishing parts: once more, scaled.  A sum too large for
        // that keeps its first value (what it misses is under 2^-110 of its
        // group's scale).
        if (__syncthreads_or((lost & 0xFFFFu) != 0)) pass(std::integral_constant<int, SPLIT_EXP>{});
    }
}

}  // namespace th
