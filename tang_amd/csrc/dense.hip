// Dense (unquantized) ComputeDevice operators, so that model code written
// against tang_compute::ComputeDevice (crates/tang-compute/src/device.rs)
// runs on this backend without a CPU round trip: matmul and its transposed /
// accumulating forms, transpose_2d, reduce_sum, bias_add, add_assign, and the
// tang-expr element-wise kernels (compiled at run time with hiprtc).
#include <hip/hiprtc.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <type_traits>
#include <vector>

#include "capi_util.hpp"
#include "ops.hpp"
#include "q8gemm.hpp"

struct th_kernel {
    th_device* dev = nullptr;
    hipModule_t module = nullptr;
    hipFunction_t fn = nullptr;
};

namespace th {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// matmul: C[m][n] (+)= op(A)[m][k] . op(B)[k][n].  A is [m][k] row-major, or
// [k][m] transposed; B is [k][n], or [n][k] transposed (device.rs:103,407,425);
// both f32 or bf16.
//
// On v_mfma_f32_16x16x32_bf16, which has sixteen times the f32 MFMA's rate: an
// f32 operand goes in as three bf16 parts (x = p0 + p1 + p2 exactly, eight bits
// each), so f32 x bf16 takes three exact products and f32 x f32 the eight whose
// parts weigh 2^-24 or more of it (the ninth is under 2^-30 of a product).  Two
// exceptions, found by each workgroup for its tile:
// - Operands or results so small that parts of them vanish: the tile is summed
//   once more with its f32 operands times 2^SPLIT_EXP.
// - A result that is not finite (an infinity times a part that is zero, a value
//   or a sum too large for that factor): summed on the f32 MFMA.
// A K of one step goes there at once (direct): the truncation inside an MFMA costs
// more than f32's roundings (from two steps on it costs less).  So does f32 x f32 of
// a shallow K in few tiles, where splitting takes longer than the slower MFMA.
//
// Workgroup: 4 waves, WGM along m; each wave TM x TN 16x16 tiles; K in steps
// of 32, both operands double-buffered in LDS as 8-value octets.  A step sums
// up by itself before it joins the accumulators (short chains of additions).
// Bound by the MFMAs and their LDS operands on large shapes, by the chain of
// steps on small ones (K split over workgroups there).  Against 64x64 tiles
// on the f32 MFMA: m 509, k 2048, n 5632, f32 x bf16 210 -> 69 us (510 TFLOP/s
// of parts; 149 if every tile holds vanishing parts, 261 if NaN); m 1, k 4096
// 275 -> 17 us; m 1024, k = n = 4096, f32 x f32 374 -> 265 us, bf16 565 -> 104 us;
// error against 64 bits 8.1e-7 -> 1.0e-7.
// ---------------------------------------------------------------------------

// An operand: `rows` rows of K values, element (row, k) at row * rs + k * ks.
struct MatOperand {
    const void* p;
    int rows;
    long rs, ks;
};

// Octet k0..k0+7 of one row, raw: bf16 pairs in a, or f32 in a and b.  vec:
// ks == 1, rows of whole dwords and the octet within K: one 16-byte load (two
// for f32) through a resource; else eight loads (clamped to the last k).
template <bool BF>
__device__ __forceinline__ void mm_load8(const MatOperand& m, const __amdgpu_buffer_rsrc_t& rs, int row0, int row, int K,
                                         int k0, bool vec, u32x4_t& a, u32x4_t& b) {
    if (vec) {
        const uint32_t off = ((uint32_t)(row - row0) * (uint32_t)m.rs + (uint32_t)k0) * (BF ? 2u : 4u);
        a = __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0);
        if constexpr (!BF) b = __builtin_amdgcn_raw_buffer_load_b128(rs, off + 16u, 0, 0);
        return;
    }
    {
        uint32_t v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const size_t at = (size_t)row * m.rs + (size_t)min(k0 + i, K - 1) * m.ks;
            v[i] = BF ? (uint32_t)((const uint16_t*)m.p)[at] : ((const uint32_t*)m.p)[at];
        }
        if constexpr (BF) {
            a = u32x4_t{v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16), v[6] | (v[7] << 16)};
        } else {
            a = u32x4_t{v[0], v[1], v[2], v[3]};
            b = u32x4_t{v[4], v[5], v[6], v[7]};
        }
    }
}

// Values at k >= K (n of the eight are real) to zero.
template <bool BF>
__device__ __forceinline__ void mm_mask(int n, u32x4_t& a, u32x4_t& b) {
    if (n >= 8) return;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if constexpr (BF) {
            a[i] = 2 * i + 1 < n ? a[i] : 2 * i < n ? a[i] & 0xFFFFu : 0u;
        } else {
            a[i] = i < n ? a[i] : 0u;
            b[i] = i + 4 < n ? b[i] : 0u;
        }
    }
}

// Value e of an octet that mm_load8 loaded.
template <bool BF>
__device__ __forceinline__ float mm_value(int e, const u32x4_t& a, const u32x4_t& b) {
    if constexpr (BF) return __uint_as_float(e & 1 ? a[e >> 1] & 0xFFFF0000u : a[e >> 1] << 16);
    else return __uint_as_float(e < 4 ? a[e] : b[e - 4]);
}

constexpr int MM_LD = 17;  // octet stride in 16-byte units (16 rows + 1: spreads the banks)

template <bool ABF, bool BBF, bool AV, bool BV, int TM, int TN, int WGM>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void matmul_kernel(
    MatOperand A, MatOperand B, float* __restrict__ c, int K, size_t split_stride, int k_per_split, int direct,
    int accumulate) {
    constexpr int PA = ABF ? 1 : 3, PB = BBF ? 1 : 3, WGN = 4 / WGM;
    constexpr bool PARTS = PA * PB > 1;
    constexpr int MB = WGM * TM, NB = WGN * TN;           // 16-row blocks of the workgroup
    constexpr int APL = MB * 4 * MM_LD, BPL = NB * 4 * MM_LD;  // one part of a step
    constexpr int AO = MB * 64, BO = NB * 64;             // octets of a step
    constexpr int AT = (AO + 255) / 256, BT = (BO + 255) / 256;
    __shared__ uint4 lds[2][PA * APL + PB * BPL];
    int bx = blockIdx.x, by = blockIdx.y, split = blockIdx.z;
    gemm_xcd_tile(bx, by, split);
    int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int q = lane >> 4, r = lane & 15;
    const int m0 = by * MB * 16, n0 = bx * NB * 16;
    const int wm = (wave / WGN) * TM, wn = (wave % WGN) * TN;
    const int kb = split * k_per_split, ke = min(K, kb + k_per_split);
    // resources based at the block's first row (offsets stay 32-bit)
    auto rsrc = [&](const MatOperand& m, int row0, size_t es) {
        const size_t left = ((size_t)(m.rows - 1 - row0) * m.rs + K) * es;  // (one row: rs need not be K)
        return buffer_rsrc((const char*)m.p + (size_t)row0 * m.rs * es, (uint32_t)min(left, (size_t)0x7FFFFFF0));
    };
    const __amdgpu_buffer_rsrc_t ars = rsrc(A, AV ? m0 : 0, ABF ? 2 : 4), brs = rsrc(B, BV ? n0 : 0, BBF ? 2 : 4);

    // octet idx of a step: (row, octet) with the index that is contiguous in
    // memory running fastest over the threads
    auto place = [](int idx, int rows, bool vec, int& row, int& o) {
        row = vec ? idx >> 2 : idx % rows;
        o = vec ? idx & 3 : idx / rows;
    };
    u32x4_t ra[AT][2], rb[BT][2];
    auto load = [&](int k) {
        const bool whole = k + 32 <= K;  // uniform: all but the last step
#pragma unroll
        for (int i = 0; i < AT; i++) {
            int row, o;
            place(min(tid + 256 * i, AO - 1), MB * 16, AV, row, o);
            mm_load8<ABF>(A, ars, m0, min(m0 + row, A.rows - 1), K, k + o * 8, AV && whole, ra[i][0], ra[i][1]);
        }
#pragma unroll
        for (int i = 0; i < BT; i++) {
            int row, o;
            place(min(tid + 256 * i, BO - 1), NB * 16, BV, row, o);
            mm_load8<BBF>(B, brs, n0, min(n0 + row, B.rows - 1), K, k + o * 8, BV && whole, rb[i][0], rb[i][1]);
        }
    };
    uint32_t lost = 0;
    auto put = [&](auto ex, auto bf, uint4* dst, int plane, int row, int o, u32x4_t (&v)[2], int k) {
        constexpr bool BF = decltype(bf)::value;
        mm_mask<BF>(K - (k + o * 8), v[0], v[1]);
        dst += ((row >> 4) * 4 + o) * MM_LD + (row & 15);
        if constexpr (BF) {
            *dst = __builtin_bit_cast(uint4, v[0]);
        } else {
            uint4 p[3];
            split3_bf16<decltype(ex)::value>(__builtin_bit_cast(uint4, v[0]), __builtin_bit_cast(uint4, v[1]), p, lost);
#pragma unroll
            for (int e = 0; e < 3; e++) dst[e * plane] = p[e];
        }
    };
    auto store = [&](auto ex, uint4* t, int k) {
#pragma unroll
        for (int i = 0; i < AT; i++) {
            int row, o;
            place(tid + 256 * i, MB * 16, AV, row, o);
            if (AO % 256 == 0 || tid + 256 * i < AO) put(ex, std::integral_constant<bool, ABF>{}, t, APL, row, o, ra[i], k);
        }
#pragma unroll
        for (int i = 0; i < BT; i++) {
            int row, o;
            place(tid + 256 * i, NB * 16, BV, row, o);
            if (BO % 256 == 0 || tid + 256 * i < BO)
                put(ex, std::integral_constant<bool, BBF>{}, t + PA * APL, BPL, row, o, rb[i], k);
        }
    };
    f32x4_t acc[TM][TN];
    auto sum = [&](auto ex) {  // f32 operands times 2^ex
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        load(kb);
        store(ex, lds[0], kb);
        __syncthreads();
        int buf = 0;
        for (int k = kb; k < ke; k += 32) {
            const uint4 *ta = lds[buf], *tb = ta + PA * APL;
            const bool more = k + 32 < ke;
            if (more) load(k + 32);
            bf16x8_t bv[TN][PB];
#pragma unroll
            for (int j = 0; j < TN; j++)
#pragma unroll
                for (int p = 0; p < PB; p++)
                    bv[j][p] = __builtin_bit_cast(bf16x8_t, tb[p * BPL + ((wn + j) * 4 + q) * MM_LD + r]);
#pragma unroll
            for (int i = 0; i < TM; i++) {
                bf16x8_t av[PA];
#pragma unroll
                for (int p = 0; p < PA; p++)
                    av[p] = __builtin_bit_cast(bf16x8_t, ta[p * APL + ((wm + i) * 4 + q) * MM_LD + r]);
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    // D = (rows of B) x (rows of A): a lane holds four consecutive n of one m
                    f32x4_t d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int w = 3; w >= 0; w--)  // the smallest products first
#pragma unroll
                        for (int p = 0; p <= w; p++)
                            if (p < PA && w - p < PB)
                                d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bv[j][w - p], av[p], d, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 4; e++) acc[i][j][e] += d[e];
                }
            }
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) mfma_pin(acc[i][j]);
            buf ^= 1;
            if (more) store(ex, lds[buf], k + 32);
            __syncthreads();
        }
    };
    // the same on the f32 MFMA, straight from memory: lane (q, r) takes octet q of row r
    auto sum_f32 = [&]() {
#pragma unroll
        for (int i = 0; i < TM; i++)
#pragma unroll
            for (int j = 0; j < TN; j++) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        for (int k = kb; k < ke; k += 32) {
            const bool whole = k + 32 <= K;
            const int k0 = k + 8 * q;
            u32x4_t a[TM][2], b[TN][2];
#pragma unroll
            for (int i = 0; i < TM; i++)
                mm_load8<ABF>(A, ars, m0, min(m0 + (wm + i) * 16 + r, A.rows - 1), K, k0, AV && whole, a[i][0], a[i][1]);
#pragma unroll
            for (int j = 0; j < TN; j++)
                mm_load8<BBF>(B, brs, n0, min(n0 + (wn + j) * 16 + r, B.rows - 1), K, k0, BV && whole, b[j][0], b[j][1]);
#pragma unroll
            for (int i = 0; i < TM; i++) mm_mask<ABF>(ke - k0, a[i][0], a[i][1]);
#pragma unroll
            for (int j = 0; j < TN; j++) mm_mask<BBF>(ke - k0, b[j][0], b[j][1]);
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++) {
                    f32x4_t d = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        d = __builtin_amdgcn_mfma_f32_16x16x4f32(mm_value<BBF>(e, b[j][0], b[j][1]),
                                                                 mm_value<ABF>(e, a[i][0], a[i][1]), d, 0, 0, 0);
                    acc[i][j] += d;
                    mfma_pin(acc[i][j]);
                }
        }
    };
    if constexpr (!PARTS) {
        sum(std::integral_constant<int, 0>{});
    } else if (direct) {
        sum_f32();
    } else {
        sum(std::integral_constant<int, 0>{});
        auto any = [&](auto test) {
            bool t = false;
#pragma unroll
            for (int i = 0; i < TM; i++)
#pragma unroll
                for (int j = 0; j < TN; j++)
#pragma unroll
                    for (int e = 0; e < 4; e++) t |= test(fabsf(acc[i][j][e]));
            return t;
        };
        const auto nonfinite = [](float v) { return !(v <= 3.402823466e38f); };
        // parts of an operand or of a product below the formats' smallest numbers
        const bool vanished = (lost & 0xFFFFu) != 0 || any([](float v) { return v > 0.0f && v < 0x1p-100f; });
        if (__syncthreads_or(vanished || any(nonfinite))) {
            if (__syncthreads_or(vanished)) {
                asm volatile("" : "+v"(tid));  // places are formed again, not kept through the first pass
                sum(std::integral_constant<int, SPLIT_EXP>{});
#pragma unroll
                for (int i = 0; i < TM; i++)
#pragma unroll
                    for (int j = 0; j < TN; j++)
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            acc[i][j][e] = __builtin_amdgcn_ldexpf(acc[i][j][e], -SPLIT_EXP * (!ABF + !BBF));
            }
            if (__syncthreads_or(any(nonfinite))) sum_f32();
        }
    }
    float* cb = c + (size_t)split * split_stride;
    const int N = B.rows;
#pragma unroll
    for (int i = 0; i < TM; i++) {
        const int m = m0 + (wm + i) * 16 + r;
        if (m >= A.rows) continue;
#pragma unroll
        for (int j = 0; j < TN; j++) {
            const int n = n0 + (wn + j) * 16 + 4 * q;
            float* p = cb + (size_t)m * N + n;
            if (N % 4 == 0 && n < N) {
                f32x4_t v = acc[i][j];
                if (accumulate) v = *(const f32x4_t*)p + v;
                *(f32x4_t*)p = v;
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (n + e < N) p[e] = accumulate ? p[e] + acc[i][j][e] : acc[i][j][e];
            }
        }
    }
}

// f32 x f32 of a shallow K over more tiles than the CUs: 64x64 tiles on the f32
// MFMA, four waves of 32x32, K in steps of 16 through LDS rows padded to 68 floats
// (the operand reads hit distinct banks).  Splitting the operands would take longer
// than the MFMAs save (matmul_dispatch has the line).
constexpr int MF_T = 64, MF_K = 16, MF_LD = MF_T + 4;

template <bool TA, bool TB>
__global__ __launch_bounds__(256) void matmul_f32_kernel(const float* __restrict__ a, const float* __restrict__ b,
                                                         float* __restrict__ c, int M, int N, int K, int accumulate) {
    __shared__ float As[MF_K][MF_LD];  // As[kk][row]
    __shared__ float Bs[MF_K][MF_LD];  // Bs[kk][col]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = blockIdx.y * MF_T, n0 = blockIdx.x * MF_T;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    f32x4_t acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // staging: each thread moves 4 elements of each 64x16 tile; the fast
    // index follows the contiguous dimension of the source
    auto stage = [&](int k0, float ra[4], float rb[4]) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int e = tid + 256 * u;
            int row, kk;
            if (TA) { row = e & 63; kk = e >> 6; }   // A[k][m]: m contiguous
            else { kk = e & 15; row = e >> 4; }      // A[m][k]: k contiguous
            const int gm = m0 + row, gk = k0 + kk;
            ra[u] = (gm < M && gk < K) ? a[TA ? (size_t)gk * M + gm : (size_t)gm * K + gk] : 0.0f;
            int col, kb;
            if (TB) { kb = e & 15; col = e >> 4; }   // B[n][k]: k contiguous
            else { col = e & 63; kb = e >> 6; }      // B[k][n]: n contiguous
            const int gn = n0 + col, gkb = k0 + kb;
            rb[u] = (gn < N && gkb < K) ? b[TB ? (size_t)gn * K + gkb : (size_t)gkb * N + gn] : 0.0f;
        }
    };
    auto store = [&](const float ra[4], const float rb[4]) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int e = tid + 256 * u;
            if (TA) As[e >> 6][e & 63] = ra[u];
            else As[e & 15][e >> 4] = ra[u];
            if (TB) Bs[e & 15][e >> 4] = rb[u];
            else Bs[e >> 6][e & 63] = rb[u];
        }
    };
    float ra[4], rb[4];
    stage(0, ra, rb);
    for (int k0 = 0; k0 < K; k0 += MF_K) {
        store(ra, rb);
        __syncthreads();
        if (k0 + MF_K < K) stage(k0 + MF_K, ra, rb);  // next tile's loads in flight during the MFMAs
#pragma unroll
        for (int ks = 0; ks < MF_K; ks += 4) {
            // 16x16x4: lane (g, r) supplies A[row r][k g] and B[k g][col r]
            const int g = lane >> 4, r = lane & 15;
            float av[2], bv[2];
#pragma unroll
            for (int i = 0; i < 2; i++) av[i] = As[ks + g][wm + 16 * i + r];
#pragma unroll
            for (int j = 0; j < 2; j++) bv[j] = Bs[ks + g][wn + 16 * j + r];
#pragma unroll
            for (int i = 0; i < 2; i++)
#pragma unroll
                for (int j = 0; j < 2; j++) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[i], bv[j], acc[i][j], 0, 0, 0);
        }
        __syncthreads();
    }
    mfma_settle(acc);
    // D: lane (g, r) holds rows 4g..4g+3 of column r
    const int g = lane >> 4, r = lane & 15;
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int col = n0 + wn + 16 * j + r;
            if (col >= N) continue;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int row = m0 + wm + 16 * i + 4 * g + e;
                if (row < M) {
                    float* p = c + (size_t)row * N + col;
                    *p = accumulate ? *p + acc[i][j][e] : acc[i][j][e];
                }
            }
        }
}

template <bool ABF, bool BBF, bool AV, bool BV, int TM, int TN, int WGM>
static void matmul_launch(const MatOperand& A, const MatOperand& B, float* c, size_t k, int acc, th_device* dev) {
    const size_t m = A.rows, n = B.rows, part = m * n * sizeof(float), cus = dev->num_cus;
    const unsigned gx = (unsigned)ceil_div(n, (size_t)(4 / WGM * TN * 16)), gy = (unsigned)ceil_div(m, (size_t)(WGM * TM * 16));
    // Split K where the tiles leave CUs idle: two workgroups per CU, each
    // split at least 128 deep.
    size_t ks = workspace_splits(dev, std::min({2 * cus / ((size_t)gx * gy), k / 128, (size_t)16}), part, dev->stream);
    const size_t per = round_up(ceil_div(k, ks), (size_t)32);
    ks = ceil_div(k, per);
    float* out = ks > 1 ? (float*)device_scratch(dev, ks * part) : c;
    // (us, parts / direct, 16 x 64 tiles: 33 x 216 x 2866, 135 workgroups, 9.2 / 6.6; 300 x
    // 300 x 1000, 304, 12.9 / 9.9; 300 x 200 x 4000, 1197, 16.9 / 20.4)
    const bool direct = k <= 32 || (!ABF && !BBF && TM == 1 && k <= 320 && (size_t)gx * gy <= 2 * cus);
    TH_LAUNCH((matmul_kernel<ABF, BBF, AV, BV, TM, TN, WGM>), dim3(gx, gy, (unsigned)ks), dim3(256), 0, dev->stream, A, B,
              out, (int)k, m * n, (int)per, (int)direct, ks > 1 ? 0 : acc);
    TH_LAUNCH_CHECK();
    if (ks > 1) launch_splitk_reduce(out, c, m, n, n, ks, acc != 0, dev->stream);
}

template <bool ABF, bool BBF, bool AV, bool BV>
static void matmul_shape(const MatOperand& A, const MatOperand& B, float* c, size_t k, int acc, th_device* dev) {
    // 16 x 64 tiles up to 16 rows and where 64 x 128 ones, their K split, come to half
    // the CUs or fewer: more workgroups, each with less to split and stage a step
    // (us, 16 x 64 / 64 x 128, f32 x bf16: 64 x 1024 x 1024, 64 workgroups, 10.6 / 12.7;
    // 100 x 576 x 1536, 96, 10.1 / 12.3; 100 x 100 x 8192, 128, 7.9 / 8.9; 300 x 100 x 4000,
    // 160, 9.2 / 9.4; 40 x 4096 x 1536, 192, 19.3 / 18.5; 128 x 2048 x 2048, 512, 26.2 / 21.3).
    const size_t large = ceil_div(A.rows, (size_t)64) * ceil_div(B.rows, (size_t)128) * std::clamp<size_t>(k / 128, 1, 16);
    if (A.rows <= 16 || 2 * large <= (size_t)dev->num_cus) matmul_launch<ABF, BBF, AV, BV, 1, 1, 1>(A, B, c, k, acc, dev);
    else matmul_launch<ABF, BBF, AV, BV, 2, 4, 2>(A, B, c, k, acc, dev);
}

template <bool ABF, bool BBF>
static void matmul_dispatch(const MatOperand& A, const MatOperand& B, float* c, size_t k, bool trans_a, bool trans_b,
                            int acc, th_device* dev) {
    // one 16-byte load per octet where k is contiguous, rows are whole dwords
    // and a block's offsets fit 32 bits
    auto vec = [](const MatOperand& m, bool bf) { return m.ks == 1 && (!bf || m.rs % 2 == 0) && m.rs <= (1l << 21); };
    const bool av = vec(A, ABF), bv = vec(B, BBF);
    if constexpr (!ABF && !BBF) {
        // us, 64x64 on the f32 MFMA / parts: 100 x 100 x 8192 7.6 / 10.0, k 160 9.5 / 10.4, k
        // 256 13.3 / 14.8; 300 x 200 x 4000 15.2 / 16.9; 1024 x 64 x 1024 5.8 / 6.6; but 512 x 128 x
        // 512 (16 x 64 tiles, direct) 7.8 / 4.7, 1000 x 200 x 200 10.9 / 6.5
        const size_t gx = ceil_div(B.rows, (size_t)MF_T), gy = ceil_div(A.rows, (size_t)MF_T);
        if (A.rows > 16 && k <= 256 && 2 * gx * gy > (size_t)dev->num_cus) {
            auto f32 = [&](auto ta, auto tb) {
                TH_LAUNCH((matmul_f32_kernel<decltype(ta)::value, decltype(tb)::value>), dim3((unsigned)gx, (unsigned)gy),
                          dim3(256), 0, dev->stream, (const float*)A.p, (const float*)B.p, c, A.rows, B.rows, (int)k, acc);
                TH_LAUNCH_CHECK();
            };
            const std::true_type t;
            const std::false_type n;
            if (trans_a && trans_b) f32(t, t);
            else if (trans_a) f32(t, n);
            else if (trans_b) f32(n, t);
            else f32(n, n);
            return;
        }
    }
    if (av && bv) matmul_shape<ABF, BBF, true, true>(A, B, c, k, acc, dev);
    else if (av) matmul_shape<ABF, BBF, true, false>(A, B, c, k, acc, dev);
    else if (bv) matmul_shape<ABF, BBF, false, true>(A, B, c, k, acc, dev);
    else matmul_shape<ABF, BBF, false, false>(A, B, c, k, acc, dev);
}

// ---------------------------------------------------------------------------
// transpose_2d (cpu.rs:317-326): out[c][r] = in[r][c], 32x32 LDS tiles.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void transpose_kernel(const float* __restrict__ in, float* __restrict__ out, int rows,
                                                        int cols) {
    __shared__ float t[32][33];
    const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int y = ty; y < 32; y += 8)
        if (r0 + y < rows && c0 + tx < cols) t[y][tx] = in[(size_t)(r0 + y) * cols + c0 + tx];
    __syncthreads();
    for (int y = ty; y < 32; y += 8)
        if (c0 + y < cols && r0 + tx < rows) out[(size_t)(c0 + y) * rows + r0 + tx] = t[tx][y];
}

// ---------------------------------------------------------------------------
// reduce_sum (cpu.rs:169-199): out[o][i] = sum over a of in[o][a][i], added
// in order a = 0, 1, ... in f32 from 0 (bit-identical to the reference).
// One thread per output; neighbouring threads read neighbouring i.
// ---------------------------------------------------------------------------
__global__ void reduce_sum_kernel(const float* __restrict__ in, float* __restrict__ out, size_t outer, size_t len,
                                  size_t inner, int accumulate) {
    const size_t total = outer * inner;
    for (size_t idx = blockIdx.x * (size_t)blockDim.x + threadIdx.x; idx < total; idx += (size_t)gridDim.x * blockDim.x) {
        const size_t o = idx / inner, i = idx - o * inner;
        const float* p = in + o * len * inner + i;
        float s = 0.0f;
        for (size_t a = 0; a < len; a++) s += p[a * inner];
        out[idx] = accumulate ? out[idx] + s : s;
    }
}

// bias_add (device.rs:378-386): out[i] = matrix[i] + bias[i % dim].
__global__ void bias_add_kernel(const float* __restrict__ m, const float* __restrict__ bias, float* __restrict__ out,
                                size_t numel, size_t dim) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < numel; i += (size_t)gridDim.x * blockDim.x)
        out[i] = m[i] + bias[i % dim];
}

// add_assign (cpu.rs:650-655): dst[i] += src[i].
__global__ void add_assign_kernel(float* __restrict__ dst, const float* __restrict__ src, size_t n) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x)
        dst[i] = dst[i] + src[i];
}

static unsigned grid_of(size_t n) { return (unsigned)std::max<size_t>(1, std::min<size_t>(ceil_div(n, 256), 8192)); }

}  // namespace th

using namespace th;

extern "C" {

int th_matmul_ex(th_device* dev, const th_buffer* a, const th_buffer* b, size_t m, size_t k, size_t n, int trans_a,
                 int trans_b, int accumulate, th_buffer* c) {
    TH_API_BEGIN
    TH_REQUIRE(dev && a && b && c, "null argument");
    TH_REQUIRE(a->dtype == TH_F32 || a->dtype == TH_BF16, "a must be f32 or bf16");
    TH_REQUIRE(b->dtype == TH_F32 || b->dtype == TH_BF16, "b must be f32 or bf16");
    require_len_any(a, m * k, "a");
    require_len_any(b, k * n, "b");
    require_len(c, TH_F32, m * n, "c");
    TH_REQUIRE(m < (1u << 31) / 64 && n < (1u << 31) / 64 && k < (1u << 31), "matmul: dimension too large");
    if (m == 0 || n == 0) return TH_OK;
    if (k == 0) {  // an empty sum: C = 0 (or C unchanged when accumulating)
        if (!accumulate) check_status(th_buffer_zero(c));
        return TH_OK;
    }
    const MatOperand A{a->ptr, (int)m, trans_a ? 1l : (long)k, trans_a ? (long)m : 1l};
    const MatOperand B{b->ptr, (int)n, trans_b ? (long)k : 1l, trans_b ? 1l : (long)n};
    float* out = (float*)c->ptr;
    const bool abf = a->dtype == TH_BF16, bbf = b->dtype == TH_BF16;
    if (abf && bbf) matmul_dispatch<true, true>(A, B, out, k, trans_a != 0, trans_b != 0, accumulate, dev);
    else if (abf) matmul_dispatch<true, false>(A, B, out, k, trans_a != 0, trans_b != 0, accumulate, dev);
    else if (bbf) matmul_dispatch<false, true>(A, B, out, k, trans_a != 0, trans_b != 0, accumulate, dev);
    else matmul_dispatch<false, false>(A, B, out, k, trans_a != 0, trans_b != 0, accumulate, dev);
    TH_API_END
}

int th_matmul(th_device* dev, const th_buffer* a, const th_buffer* b, size_t m, size_t k, size_t n, th_buffer* c) {
    return th_matmul_ex(dev, a, b, m, k, n, 0, 0, 0, c);
}

int th_matmul_b_transposed(th_device* dev, const th_buffer* a, const th_buffer* b, size_t m, size_t k, size_t n,
                           th_buffer* c) {
    return th_matmul_ex(dev, a, b, m, k, n, 0, 1, 0, c);
}

int th_transpose_2d(th_device* dev, const th_buffer* in, size_t rows, size_t cols, th_buffer* out) {
    TH_API_BEGIN
    TH_REQUIRE(dev && in && out, "null argument");
    require_len(in, TH_F32, rows * cols, "in");
    require_len(out, TH_F32, rows * cols, "out");
    TH_REQUIRE(rows < (1u << 31) && cols < (1u << 31), "transpose: dimension too large");
    if (rows == 0 || cols == 0) return TH_OK;
    TH_REQUIRE(ceil_div(rows, 32) < 65536, "transpose: more than 2^21 rows");
    TH_LAUNCH(transpose_kernel, dim3((unsigned)ceil_div(cols, 32), (unsigned)ceil_div(rows, 32)), dim3(256), 0,
                       dev->stream, (const float*)in->ptr, (float*)out->ptr, (int)rows, (int)cols);
    TH_LAUNCH_CHECK();
    TH_API_END
}

int th_reduce_sum(th_device* dev, const th_buffer* in, const size_t* shape, size_t ndim, size_t axis, int accumulate,
                  th_buffer* out) {
    TH_API_BEGIN
    TH_REQUIRE(dev && in && out && (shape || ndim == 0), "null argument");
    TH_REQUIRE(axis < ndim, "reduce_sum: axis out of range");
    size_t outer = 1, inner = 1;
    for (size_t i = 0; i < axis; i++) outer *= shape[i];
    for (size_t i = axis + 1; i < ndim; i++) inner *= shape[i];
    const size_t len = shape[axis];
    require_len(in, TH_F32, outer * len * inner, "in");
    require_len(out, TH_F32, outer * inner, "out");
    if (outer * inner == 0) return TH_OK;
    TH_LAUNCH(reduce_sum_kernel, dim3(grid_of(outer * inner)), dim3(256), 0, dev->stream,
                       (const float*)in->ptr, (float*)out->ptr, outer, len, inner, accumulate);
    TH_LAUNCH_CHECK();
    TH_API_END
}

int th_bias_add(th_device* dev, const th_buffer* matrix, const th_buffer* bias, size_t numel, size_t dim,
                th_buffer* out) {
    TH_API_BEGIN
    TH_REQUIRE(dev && matrix && bias && out, "null argument");
    TH_REQUIRE(dim > 0 || numel == 0, "bias_add: dim is 0");
    require_len(matrix, TH_F32, numel, "matrix");
    require_len(bias, TH_F32, dim, "bias");
    require_len(out, TH_F32, numel, "out");
    if (numel == 0) return TH_OK;
    TH_LAUNCH(bias_add_kernel, dim3(grid_of(numel)), dim3(256), 0, dev->stream, (const float*)matrix->ptr,
                       (const float*)bias->ptr, (float*)out->ptr, numel, dim);
    TH_LAUNCH_CHECK();
    TH_API_END
}

int th_add_assign(th_device* dev, th_buffer* dst, const th_buffer* src) {
    TH_API_BEGIN
    TH_REQUIRE(dev && dst && src, "null argument");
    TH_REQUIRE(dst->dtype == TH_F32 && src->dtype == TH_F32, "add_assign: f32 buffers");
    TH_REQUIRE(dst->n == src->n, "add_assign: lengths differ");  // cpu.rs:651 asserts equal lengths
    if (dst->n == 0) return TH_OK;
    TH_LAUNCH(add_assign_kernel, dim3(grid_of(dst->n)), dim3(256), 0, dev->stream, (float*)dst->ptr,
                       (const float*)src->ptr, dst->n);
    TH_LAUNCH_CHECK();
    TH_API_END
}

// ---- run-time compiled element-wise kernels --------------------------------

int th_kernel_compile(th_device* dev, const char* source, const char* entry, th_kernel** out) {
    TH_API_BEGIN
    TH_REQUIRE(dev && source && entry && out, "null argument");
    hiprtcProgram prog;
    if (hiprtcCreateProgram(&prog, source, "elementwise.hip", 0, nullptr, nullptr) != HIPRTC_SUCCESS)
        throw Error(TH_ERR_HIP, "hiprtcCreateProgram failed");
    // gfx950 only; no packed-FP32 instructions and no FMA contraction, as
    // the library's own kernels
    const char* opts[] = {"--offload-arch=gfx950", "-O3", "-ffp-contract=off", "-Xclang", "-target-feature",
                          "-Xclang", "-packed-fp32-ops"};
    const hiprtcResult rc = hiprtcCompileProgram(prog, (int)(sizeof(opts) / sizeof(opts[0])), opts);
    if (rc != HIPRTC_SUCCESS) {
        size_t n = 0;
        std::string log;
        if (hiprtcGetProgramLogSize(prog, &n) == HIPRTC_SUCCESS && n > 1) {
            log.resize(n);
            hiprtcGetProgramLog(prog, &log[0]);
        }
        hiprtcDestroyProgram(&prog);
        throw Error(TH_ERR_INVALID, std::string("kernel compile failed: ") + hiprtcGetErrorString(rc) + "\n" + log);
    }
    size_t code_size = 0;
    hiprtcGetCodeSize(prog, &code_size);
    std::vector<char> code(code_size);
    hiprtcGetCode(prog, code.data());
    hiprtcDestroyProgram(&prog);
    th_kernel* k = new th_kernel();
    k->dev = dev;
    hipError_t e = hipModuleLoadData(&k->module, code.data());
    if (e == hipSuccess) e = hipModuleGetFunction(&k->fn, k->module, entry);
    if (e != hipSuccess) {
        if (k->module) (void)hipModuleUnload(k->module);
        delete k;
        throw Error(TH_ERR_HIP, std::string("module load: ") + hipGetErrorString(e));
    }
    device_retain(dev);
    *out = k;
    TH_API_END
}

int th_kernel_free(th_kernel* k) {
    TH_API_BEGIN
    if (!k) return TH_OK;
    th_device* d = k->dev;
    device_drain(d);
    (void)hipModuleUnload(k->module);
    delete k;
    device_release(d);
    TH_API_END
}

int th_elementwise(th_kernel* k, const th_buffer* const* inputs, size_t n_inputs, size_t numel, th_buffer* out) {
    TH_API_BEGIN
    TH_REQUIRE(k && out && (inputs || n_inputs == 0), "null argument");
    TH_REQUIRE(n_inputs <= 64, "elementwise: at most 64 inputs");
    TH_REQUIRE(numel <= 0xFFFFFFFFu, "elementwise: count is a 32-bit kernel argument");
    for (size_t i = 0; i < n_inputs; i++) require_len(inputs[i], TH_F32, numel, "input");
    require_len(out, TH_F32, numel, "out");
    if (numel == 0) return TH_OK;
    // argument block of the generated signature: in0..in{n-1}, outputs, count
    std::vector<char> args;
    auto put = [&](const void* p, size_t sz, size_t align) {
        args.resize(round_up(args.size(), align));
        const size_t o = args.size();
        args.resize(o + sz);
        std::memcpy(&args[o], p, sz);
    };
    for (size_t i = 0; i < n_inputs; i++) put(&inputs[i]->ptr, sizeof(void*), sizeof(void*));
    put(&out->ptr, sizeof(void*), sizeof(void*));
    const unsigned count = (unsigned)numel;
    put(&count, sizeof(count), sizeof(count));
    size_t bytes = args.size();
    void* cfg[] = {HIP_LAUNCH_PARAM_BUFFER_POINTER, args.data(), HIP_LAUNCH_PARAM_BUFFER_SIZE, &bytes,
                   HIP_LAUNCH_PARAM_END};
    TH_HIP(hipModuleLaunchKernel(k->fn, (unsigned)ceil_div(numel, 256), 1, 1, 256, 1, 1, 0, k->dev->stream, nullptr,
                                 cfg));
    TH_API_END
}

}  // extern "C"
