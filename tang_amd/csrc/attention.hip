// KV-cached decode attention: ComputeDevice::kv_attention
// (crates/tang-compute/src/cpu.rs:257-315).  Query i of q_len attends to cache
// positions 0..cache_start+i; GQA maps head h to kv head h/(n_heads/n_kv_heads);
// scores are scaled by 1/sqrt(head_dim); f32 arithmetic throughout.
//
// Split-K ("flash-decoding") form: each workgroup scores one chunk of
// positions for one (query, head), keeps the chunk's max m, sum l and
// unnormalised weighted V, and the last chunk of each (query, head) to finish
// merges the chunks with exp(m_s - M) weights (one launch in all).  From some
// work on head_dim 64, 128 and 256 run on MFMA with the query heads of one kv head as
// rows of one tile, so a K/V row is read once for all of them; there is no
// length cap (the reference CUDA kernel holds scores in a fixed 2048-float
// array, attention_cuda.rs:85).  Scores, softmax and sums are f32: with an f16
// cache the f32 operand of each product goes in as three f16 parts, which hold
// all 24 bits of a value down to 2^-26 of the row's largest (AttnParts); with an
// f32 cache the products run on the f32 MFMA.  An MFMA truncates what it adds to
// a larger sum, so sums stay short and meet in plain additions.
#include <algorithm>
#include <mutex>
#include <type_traits>

#include "attention.hpp"
#include "capi_util.hpp"
#include "ops.hpp"
#include "qlinear.hpp"

namespace th {

// Generic path for head dims without a tuned kernel: one wave per
// (query, head), online softmax in the reference's own order.
template <typename CT>
__global__ __launch_bounds__(64) void attn_generic_kernel(const float* __restrict__ q, const CT* __restrict__ kc,
                                                          const CT* __restrict__ vc, int cache_start, int n_heads,
                                                          int n_kv_heads, int head_dim, float* __restrict__ out) {
    const int h = blockIdx.x, qi = blockIdx.y, lane = threadIdx.x;
    const int total_dim = n_heads * head_dim, kv_dim = n_kv_heads * head_dim;
    const int kv_h = h / (n_heads / n_kv_heads);
    const float scale = 1.0f / sqrtf((float)head_dim);
    const float* qp = q + (size_t)qi * total_dim + h * head_dim;
    float acc[8];
    for (int i = 0; i < 8; i++) acc[i] = 0.0f;
    float rmax = -INFINITY, rsum = 0.0f;
    const int attend = cache_start + qi + 1;
    for (int j = 0; j < attend; j++) {
        const CT* kr = kc + (size_t)j * kv_dim + kv_h * head_dim;
        float part = 0.0f;
        for (int i = 0, d = lane; d < head_dim; i++, d += 64) part += qp[d] * (float)kr[d];
        const float score = wave_sum(part) * scale;
        const float nmax = fmaxf(rmax, score);
        const float es = expf(score - nmax), rs = expf(rmax - nmax);
        rsum = rsum * rs + es;
        const CT* vr = vc + (size_t)j * kv_dim + kv_h * head_dim;
        for (int i = 0, d = lane; d < head_dim; i++, d += 64) acc[i] = acc[i] * rs + es * (float)vr[d];
        rmax = nmax;
    }
    const float inv = 1.0f / rsum;
    for (int i = 0, d = lane; d < head_dim; i++, d += 64) out[(size_t)qi * total_dim + h * head_dim + d] = acc[i] * inv;
}

// One row (query, head) over some keys by one wave in plain f32, for the rows
// whose MFMA sums are not finite (an infinity times a part that is zero is NaN, and
// a block's later keys carry weight zero rather than being left out): blocks of
// `block` keys every `step` from `from` on, up to `to`.  D / 8 lanes share a key;
// the wave's keys meet at the end, when lane e holds sums of dims 8e..8e+7.
struct AttnRow {
    float m, l, acc[8];
};
template <int D, typename CT>
__device__ __noinline__ AttnRow attn_row_plain(const float* __restrict__ q, const CT* __restrict__ kc,
                                               const CT* __restrict__ vc, int kv_dim, int from, int to, int block, int step,
                                               int lane) {
    constexpr int LPK = D / 8, KPW = 64 / LPK, U = sizeof(CT) == 2 ? 4 : 2;
    const int slot = lane / LPK, e = lane % LPK;
    const float scale = 1.0f / sqrtf((float)D);
    float qv[8];
    AttnRow x;
    x.m = -INFINITY;
    x.l = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        qv[i] = q[e * 8 + i];
        x.acc[i] = 0.0f;
    }
    bool nan = false;  // a NaN score: so is every output
    for (int base = from; base < to && !nan; base += step) {
        const int end = min(to, base + block);
        for (int j0 = base; j0 < end && !nan; j0 += KPW * U) {
            float k[U][8], v[U][8];
#pragma unroll
            for (int u = 0; u < U; u++) {
                const size_t at = (size_t)min(j0 + u * KPW + slot, end - 1) * kv_dim + e * 8;
                load8<CT>(kc + at, k[u]);
                load8<CT>(vc + at, v[u]);
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                float d = 0.0f;
#pragma unroll
                for (int i = 0; i < 8; i++) d += qv[i] * k[u][i];
#pragma unroll
                for (int o = LPK / 2; o > 0; o >>= 1) d += __shfl_xor(d, o, 64);
                if (j0 + u * KPW + slot >= end) continue;
                const float s = d * scale, mn = fmaxf(x.m, s), ref = mn == -INFINITY ? 0.0f : mn;
                const float p = expf(s - ref), a = expf(x.m - ref);
                x.l = x.l * a + p;
#pragma unroll
                for (int i = 0; i < 8; i++) x.acc[i] = x.acc[i] * a + p * v[u][i];
                x.m = mn;
            }
            nan = __any(x.l != x.l);
        }
    }
#pragma unroll
    for (int o = LPK; o < 64; o <<= 1) {
        const float mo = __shfl_xor(x.m, o, 64), lo = __shfl_xor(x.l, o, 64);
        const float M = fmaxf(x.m, mo), f = x.m == -INFINITY ? 0.0f : expf(x.m - M), g = mo == -INFINITY ? 0.0f : expf(mo - M);
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float ao = __shfl_xor(x.acc[i], o, 64);
            x.acc[i] = x.acc[i] * f + ao * g;
        }
        x.l = x.l * f + lo * g;
        x.m = M;
    }
    return x;
}

typedef _Float16 attn_f16x4_t __attribute__((ext_vector_type(4)));
typedef short attn_short4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) attn_short4_t attn_lds_short4_t;

// The MFMA side of one wave: 16 rows against blocks of KT 16-key tiles, both
// products transposed so that no operand is shuffled (see attn_prefill_kernel):
// S^T = K.Q^T leaves lane (g, r) the scores of row r for keys 4g..4g+3 of each
// tile, which is the B operand that O^T += V^T.P^T needs; lane (g, r)
// accumulates dims 4g..4g+3 of each 16-dim tile of row r.
// f16 cache: k octets as loaded, V^T from row-major LDS by transposing reads.
// f32 cache: v_mfma_f32_16x16x4, contraction index g of step (c, e) = dim
// 16c + 4g + e (S) and key 4g + e of a tile (P.V).
//
// The f32 operand against an f16 cache, brought to at most 2^15: x = h + 2^-11 (m
// + l), each part f16 with the eleven bits that the ones before left.  m and l
// share a factor, so what x keeps below h reaches 2^-35, and sum up apart from h.
struct AttnParts {
    _Float16 h, m, l;
    __device__ __forceinline__ explicit AttnParts(float x) {
        h = (_Float16)x;
        const float r = (x - (float)h) * 2048.0f;
        m = (_Float16)r;
        l = (_Float16)(r - (float)m);
    }
    __device__ __forceinline__ static float join(float h, float ml) { return __builtin_fmaf(ml, 1.0f / 2048.0f, h); }
};
constexpr int ATTN_TOP = 15;  // the row's largest in [2^14, 2^15)

// Sum of N values in pairs, then pairs of pairs.
template <int N>
__device__ __forceinline__ attn_f32x4_t attn_tree_sum(attn_f32x4_t (&v)[N]) {
#pragma unroll
    for (int w = 1; w < N; w *= 2)
#pragma unroll
        for (int i = 0; i + w < N; i += 2 * w) v[i] += v[i + w];
    return v[0];
}

template <int D, typename CT, int KT>
struct AttnWave {
    static constexpr bool H = sizeof(CT) == 2;
    static constexpr int NK = H ? D / 32 : D / 16;  // 16-byte pieces of a K row per lane
    static constexpr int NDT = D / 16;
    static constexpr int LD = D + (H ? 8 : 4);      // LDS row stride (elements)
    attn_f16x8_t qh[H ? NK : 1], qm[H ? NK : 1], ql[H ? NK : 1];
    attn_f32x4_t qf[H ? 1 : NK];
    attn_f32x4_t o[NDT];
    float m, l;
    int qe;

    // dims of piece c of lane group g
    __device__ __forceinline__ static int dim0(int c, int g) { return H ? c * 32 + 8 * g : c * 16 + 4 * g; }

    __device__ __forceinline__ void init(const float* qrow, int g) {
        m = -INFINITY;
        l = 0.0f;
        qe = 0;
#pragma unroll
        for (int t = 0; t < NDT; t++) o[t] = attn_f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (H) {
            float v[NK][8], mx = 0.0f;
#pragma unroll
            for (int c = 0; c < NK; c++) {
                const float4 a = *(const float4*)(qrow + dim0(c, g)), b = *(const float4*)(qrow + dim0(c, g) + 4);
                v[c][0] = a.x; v[c][1] = a.y; v[c][2] = a.z; v[c][3] = a.w;
                v[c][4] = b.x; v[c][5] = b.y; v[c][6] = b.z; v[c][7] = b.w;
#pragma unroll
                for (int i = 0; i < 8; i++) mx = fmaxf(mx, fabsf(v[c][i]));
            }
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            qe = range_exp(mx, ATTN_TOP);
#pragma unroll
            for (int c = 0; c < NK; c++)
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const AttnParts x(__builtin_amdgcn_ldexpf(v[c][i], -qe));
                    qh[c][i] = x.h;
                    qm[c][i] = x.m;
                    ql[c][i] = x.l;
                }
        } else {
#pragma unroll
            for (int c = 0; c < NK; c++) qf[c] = *(const attn_f32x4_t*)(qrow + dim0(c, g));
        }
    }

    // scores of one 16-key tile from its K pieces
    __device__ __forceinline__ attn_f32x4_t score(const attn_u32x4_t (&k)[NK]) const {
        const attn_f32x4_t z = {0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (H) {
            constexpr int CH = D > 128 ? 2 : 1;  // pieces that sum up in one chain (two: the registers end)
            attn_f32x4_t ml = z, h[NK / CH];
#pragma unroll
            for (int c = 0; c < NK; c++)
                ml = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(attn_f16x8_t, k[c]), ql[c], ml, 0, 0, 0);
#pragma unroll
            for (int c = 0; c < NK; c++)
                ml = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(attn_f16x8_t, k[c]), qm[c], ml, 0, 0, 0);
#pragma unroll
            for (int c = 0; c < NK; c++)
                h[c / CH] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(attn_f16x8_t, k[c]), qh[c],
                                                                   c % CH ? h[c / CH] : z, 0, 0, 0);
            attn_f32x4_t s = attn_tree_sum(h);
#pragma unroll
            for (int i = 0; i < 4; i++) s[i] = AttnParts::join(s[i], ml[i]);
            return s;
        } else {
            // Sums of eight products, which meet in pairs as soon as the next
            // piece's MFMAs are on their way.
            attn_f32x4_t level[5], d[2], p[2];
#pragma unroll
            for (int c = 0; c <= NK; c++) {
                if (c < NK) {
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        d[e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(attn_f32x4_t, k[c < NK ? c : 0])[e],
                                                                        qf[c < NK ? c : 0][e], e < 2 ? z : d[e & 1], 0, 0, 0);
                }
                if (c > 0) {
                    attn_f32x4_t u = p[0] + p[1];
                    int l = 0;
#pragma unroll
                    for (int n = c - 1; n & 1; n >>= 1) u = level[l++] + u;
                    level[l] = u;
                }
                p[0] = d[0];
                p[1] = d[1];
            }
            return level[NK == 4 ? 2 : NK == 8 ? 3 : 4];
        }
    }

    // the block's raw scores (key0: first key; keys past `last` of this row
    // are masked) through the online softmax; leaves probabilities in s and
    // returns the factor of the sums so far
    __device__ __forceinline__ float softmax(attn_f32x4_t (&s)[KT], int key0, int last, float scale, int g) {
        float bm = -INFINITY;
#pragma unroll
        for (int t = 0; t < KT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float v = s[t][i] * scale;
                if constexpr (H) v = __builtin_amdgcn_ldexpf(v, qe);
                if (key0 + t * 16 + 4 * g + i > last) v = -INFINITY;
                s[t][i] = v;
                bm = fmaxf(bm, v);
            }
        bm = fmaxf(bm, __shfl_xor(bm, 16, 64));
        bm = fmaxf(bm, __shfl_xor(bm, 32, 64));
        const float mn = fmaxf(m, bm), ref = mn == -INFINITY ? 0.0f : mn;  // no key of this row yet: weights 0
        const float a = expf(m - ref);
        float ps = 0.0f;
#pragma unroll
        for (int t = 0; t < KT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                s[t][i] = expf(s[t][i] - ref);
                ps += s[t][i];
            }
        l = l * a + ps;  // this lane's keys; summed over g at the end
        m = mn;
        return a;
    }

    // o = o * a + V^T.P^T over the block's V rows vs[key][LD]; the block sums
    // up by itself first (short chains of f32 additions)
    __device__ __forceinline__ void pv(const attn_f32x4_t (&p)[KT], float a, const CT* vs, int g, int r) {
        auto join = [&](int dt, const attn_f32x4_t& v) {
#pragma unroll
            for (int i = 0; i < 4; i++) o[dt][i] = __builtin_fmaf(o[dt][i], a, v[i]);
        };
        if constexpr (H) {
            constexpr int KP = (KT + 1) / 2;  // 32-key steps (an odd last tile pairs with zeros)
            attn_f16x8_t ph[KP], pm[KP], pl[KP];
#pragma unroll
            for (int c = 0; c < KP; c++)
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const int t = 2 * c + (i >> 2);
                    const AttnParts x(t < KT ? p[t < KT ? t : 0][i & 3] * 32768.0f : 0.0f);
                    ph[c][i] = x.h;
                    pm[c][i] = x.m;
                    pl[c][i] = x.l;
                }
#pragma unroll
            for (int dt = 0; dt < NDT; dt++) {
                attn_f32x4_t d = {0.0f, 0.0f, 0.0f, 0.0f}, ml = d;
#pragma unroll
                for (int c = 0; c < KP; c++) {
                    // lane r of a row group addresses four dims of key (r >> 2) and gets four keys of dim r
                    attn_short4_t v[2];
#pragma unroll
                    for (int hf = 0; hf < 2; hf++) {
                        const int key = (2 * c + (2 * c + hf < KT ? hf : 0)) * 16 + 4 * g + (r >> 2);
                        v[hf] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                            (attn_lds_short4_t*)(vs + (size_t)key * LD + dt * 16 + 4 * (r & 3)));
                    }
                    const attn_f16x4_t a0 = __builtin_bit_cast(attn_f16x4_t, v[0]), a1 = __builtin_bit_cast(attn_f16x4_t, v[1]);
                    const attn_f16x8_t va = {a0[0], a0[1], a0[2], a0[3], a1[0], a1[1], a1[2], a1[3]};
                    ml = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, pl[c], ml, 0, 0, 0);
                    ml = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, pm[c], ml, 0, 0, 0);
                    d = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, ph[c], d, 0, 0, 0);
                }
#pragma unroll
                for (int i = 0; i < 4; i++) d[i] = AttnParts::join(d[i], ml[i]);
                join(dt, d);
            }
        } else {
#pragma unroll
            for (int dt = 0; dt < NDT; dt++) {
                attn_f32x4_t d[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
                for (int t = 0; t < KT; t++)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        d[e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32((float)vs[(t * 16 + 4 * g + e) * LD + dt * 16 + r],
                                                                        p[t][e], d[e & 1], 0, 0, 0);
                join(dt, d[0] + d[1]);
            }
        }
    }

    // whether this lane's sums are (a NaN score makes l one)
    __device__ __forceinline__ bool finite() const {
        bool f = l == l;
#pragma unroll
        for (int t = 0; t < NDT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) f &= fabsf(o[t][i]) <= 3.402823466e38f;
        return f;
    }

    __device__ __forceinline__ void finish() {  // l over the row's lanes; o back from its 2^15
        l += __shfl_xor(l, 16, 64);
        l += __shfl_xor(l, 32, 64);
        if constexpr (H) {
#pragma unroll
            for (int t = 0; t < NDT; t++) o[t] *= 1.0f / 32768.0f;
        }
    }
};

// Decode: at most 16 rows (queries x heads of one kv head).  Workgroup = (kv
// head, split of `per` keys); its NW waves take KB-key blocks in turn, each
// with its own softmax state: K straight from memory into the MFMA operand,
// V through the wave's own LDS rows, no workgroup barrier until the waves'
// states merge.  Splits merge in the last one to arrive (coherent records).
// Bound by latency: one pass of loads and MFMAs (some 2.7 us), the waves'
// merge, and the record-arrival-record chain of the splits' (3.5 us).  8192
// keys, 32 heads on 8 kv heads of 128 dims, f16: 32.0 -> 16.6 us (the split
// kernel reads K and V once for each of four heads).
template <int D, typename CT>
struct AttnDec {
    static constexpr int KB = D <= 128 ? 32 : 16;  // keeps the registers, and f32's eight regions, in bounds
    typedef AttnWave<D, CT, KB / 16> Wave;
    static constexpr size_t ROWS = (size_t)KB * Wave::LD * sizeof(CT), MERGE = (size_t)16 * D * 4;
    static constexpr size_t REGION = ROWS > MERGE ? ROWS : MERGE;  // V rows, then the wave's 16 rows of sums
};

template <int D, typename CT, int NW>
__global__ __launch_bounds__(64 * NW) void attn_rows_decode_kernel(
    const float* __restrict__ q, const CT* __restrict__ kc, const CT* __restrict__ vc, int cache_start, int q_len, int G,
    int n_kv_heads, int per, int n_splits, float* __restrict__ part_o, float* __restrict__ part_ml,
    int* __restrict__ counters, float* __restrict__ out) {
    typedef AttnDec<D, CT> T;
    typedef typename T::Wave Wave;
    constexpr int KB = T::KB, KT = KB / 16;
    constexpr int CPR = D * (int)sizeof(CT) / 16, VL = KB * CPR / 64;
    extern __shared__ __align__(16) char lds[];
    __shared__ float sm[NW][16], sl[NW][16], sM[16];
    __shared__ int s_flag;
    const int kv_h = blockIdx.x, s = blockIdx.y, R = q_len * G, n_heads = n_kv_heads * G, kv_dim = n_kv_heads * D;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, r = lane & 15;
    const int row = min(r, R - 1), qi = row / G;
    const int j0 = s * per, j1 = min(cache_start + q_len, j0 + per);
    CT* vs = (CT*)(lds + wave * T::REGION);
    Wave w;
    w.init(q + ((size_t)qi * n_heads + kv_h * G + (row - qi * G)) * D, g);
    const float scale = 1.0f / sqrtf((float)D);
    const int last = min(cache_start + qi, j1 - 1);
    for (int key0 = j0 + wave * KB; key0 < j1; key0 += NW * KB) {
        attn_u32x4_t k[KT][Wave::NK], v[VL];
        // rows past the split re-read its last row (masked)
#pragma unroll
        for (int t = 0; t < KT; t++) {
            const CT* kr = kc + (size_t)min(key0 + t * 16 + r, j1 - 1) * kv_dim + kv_h * D;
#pragma unroll
            for (int c = 0; c < Wave::NK; c++) k[t][c] = *(const attn_u32x4_t*)(kr + Wave::dim0(c, g));
        }
        auto load_v = [&]() {
#pragma unroll
            for (int i = 0; i < VL; i++) {
                const int idx = lane + 64 * i;
                v[i] = *(const attn_u32x4_t*)((const char*)(vc + (size_t)min(key0 + idx / CPR, j1 - 1) * kv_dim + kv_h * D) +
                                              (idx % CPR) * 16);
            }
        };
        // every load on its way before the first is used (left alone the
        // compiler sinks V's to their stores, one wait each); with 256 dims V
        // takes the registers that K leaves
        if constexpr (D <= 128) load_v();
        __builtin_amdgcn_sched_barrier(0);
        attn_f32x4_t sc[KT];
#pragma unroll
        for (int t = 0; t < KT; t++) sc[t] = w.score(k[t]);
        if constexpr (D > 128) {
            __builtin_amdgcn_sched_barrier(0);
            load_v();
            __builtin_amdgcn_sched_barrier(0);
        }
        const float a = w.softmax(sc, key0, last, scale, g);
#pragma unroll
        for (int i = 0; i < VL; i++) {
            const int idx = lane + 64 * i;
            *(attn_u32x4_t*)((char*)(vs + (idx / CPR) * Wave::LD) + (idx % CPR) * 16) = v[i];
        }
        wave_lds_fence();
        w.pv(sc, a, vs, g, r);
        wave_lds_fence();  // the rows are rewritten by the next block
    }
    w.finish();
    float* mo = (float*)vs;  // [16][D]
#pragma unroll
    for (int t = 0; t < Wave::NDT; t++) *(attn_f32x4_t*)(mo + r * D + t * 16 + 4 * g) = w.o[t];
    if (g == 0) { sm[wave][r] = w.m; sl[wave][r] = w.l; }
    if (__any(!w.finite())) {
        wave_lds_fence();
        for (int rw = 0; rw < R; rw++) {
            const int qr = rw / G;
            const AttnRow x = attn_row_plain<D, CT>(q + ((size_t)qr * n_heads + kv_h * G + rw - qr * G) * D, kc + kv_h * D,
                                                    vc + kv_h * D, kv_dim, j0 + wave * KB, min(j1, cache_start + qr + 1), KB,
                                                    NW * KB, lane);
            if (lane < D / 8) {
#pragma unroll
                for (int i = 0; i < 8; i++) mo[rw * D + lane * 8 + i] = x.acc[i];
            }
            if (lane == 0) { sm[wave][rw] = x.m; sl[wave][rw] = x.l; }
        }
    }
    __syncthreads();
    if (tid < 16) {  // row tid: the waves' weights relative to the workgroup's maximum, and their sum
        float M = -INFINITY, L = 0.0f;
#pragma unroll
        for (int x = 0; x < NW; x++) M = fmaxf(M, sm[x][tid]);
#pragma unroll
        for (int x = 0; x < NW; x++) {
            const float f = sm[x][tid] == -INFINITY ? 0.0f : expf(sm[x][tid] - M);
            L = __builtin_fmaf(f, sl[x][tid], L);
            sm[x][tid] = f;
        }
        sM[tid] = M;
        sl[0][tid] = L;
    }
    __syncthreads();
    auto out_row = [&](int rw) { return out + ((size_t)(rw / G) * n_heads + kv_h * G + rw % G) * D; };
    for (int i = tid; i < R * D; i += 64 * NW) {
        const int rw = i / D, d = i % D;
        float A = 0.0f;
#pragma unroll
        for (int x = 0; x < NW; x++) A = __builtin_fmaf(sm[x][rw], ((const float*)(lds + x * T::REGION))[rw * D + d], A);
        if (n_splits == 1) {
            out_row(rw)[d] = A * (1.0f / sl[0][rw]);
        } else {
            const size_t rec = ((size_t)kv_h * R + rw) * n_splits + s;
            st_coherent(&part_o[rec * D + d], A);
            if (d == 0) { st_coherent(&part_ml[2 * rec], sM[rw]); st_coherent(&part_ml[2 * rec + 1], sl[0][rw]); }
        }
    }
    if (n_splits > 1) {
        if (!last_arrival(&counters[kv_h], n_splits, &s_flag)) return;
        const size_t rec0 = (size_t)kv_h * R * n_splits;
        const int recs = R * n_splits;
        const __amdgpu_buffer_rsrc_t ro = buffer_rsrc(part_o + rec0 * D, (uint32_t)(recs * D) * 4u);
        float* wt = (float*)lds;  // [R][n_splits] weights (maxima first), then the sums
        ld_coherent_to_lds<64 * NW>(part_ml + rec0 * 2, 2 * recs, wt, tid);
        // the first sums of this thread come in while the weights are formed
        constexpr int U = 16;
        float o[U];
        auto load_o = [&](int i, int c) {
#pragma unroll
            for (int u = 0; u < U; u++)  // past the last split: weight 0 below
                o[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                    ro, ((i / D * n_splits + min(c + u, n_splits - 1)) * D + i % D) * 4, 0, CPOL_SC1));
        };
        if (tid < R * D) load_o(tid, 0);
        __syncthreads();
        for (int rw = wave; rw < R; rw += NW) {  // weights exp(m - M) / L in place of the maxima
            float* wr = wt + 2 * rw * n_splits;
            float M = -INFINITY, L = 0.0f;
            for (int x = lane; x < n_splits; x += 64) M = fmaxf(M, wr[2 * x]);
            M = wave_max(M);
            for (int x = lane; x < n_splits; x += 64) {
                const float f = wr[2 * x] == -INFINITY ? 0.0f : expf(wr[2 * x] - M);
                L = __builtin_fmaf(f, wr[2 * x + 1], L);
                wr[2 * x] = f;
            }
            L = wave_sum(L);
            for (int x = lane; x < n_splits; x += 64) wr[2 * x] *= 1.0f / L;
        }
        __syncthreads();
        for (int i = tid; i < R * D; i += 64 * NW) {
            const float* wr = wt + 2 * (i / D) * n_splits;
            float A = 0.0f;
            for (int c = 0; c < n_splits; c += U) {
                if (i != tid || c > 0) load_o(i, c);
#pragma unroll
                for (int u = 0; u < U; u++)
                    if (c + u < n_splits) A = __builtin_fmaf(wr[2 * (c + u)], o[u], A);
            }
            out_row(i / D)[i % D] = A;
        }
    }
}

// More than 16 rows: workgroup = (64 rows of one kv head, kv head, split of
// the tile's key blocks); four waves of 16 rows share KB-key blocks of K and V
// in LDS, the next block's loads in flight meanwhile.  With one split the
// result goes out, else a record per row that attn_rows_merge_kernel merges.
// 384 queries behind 512 positions, 16 heads on 8 kv heads of 128 dims, f16
// cache: 240 -> 31 us (the split kernel reads every K/V row once per query).
template <int D, typename CT>
struct AttnPre {
    static constexpr int KB = 128 * 64 / D * 2 / (int)sizeof(CT) < 64 ? 128 * 64 / D * 2 / (int)sizeof(CT) : 64;
    typedef AttnWave<D, CT, KB / 16> Wave;
};

template <int D, typename CT>
__global__ __launch_bounds__(256) void attn_rows_kernel(const float* __restrict__ q, const CT* __restrict__ kc,
                                                        const CT* __restrict__ vc, int cache_start, int q_len, int G,
                                                        int n_kv_heads, int n_splits, float* __restrict__ part_o,
                                                        float* __restrict__ part_ml, float* __restrict__ out) {
    typedef AttnPre<D, CT> T;
    typedef typename T::Wave Wave;
    constexpr int KB = T::KB, KT = KB / 16, LD = Wave::LD;
    constexpr int CPR = D * (int)sizeof(CT) / 16, NL = KB * CPR / 256;
    static_assert(NL * 256 == KB * CPR, "whole pieces per thread");
    __shared__ __align__(16) CT ks[KB * LD], vs[KB * LD];
    const int kv_h = blockIdx.y, s = blockIdx.z, R = q_len * G, n_heads = n_kv_heads * G, kv_dim = n_kv_heads * D;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, r = lane & 15;
    const int w0 = blockIdx.x * 64 + wave * 16;  // this wave's first row
    const int row = min(w0 + r, R - 1), qi = row / G, h = kv_h * G + (row - qi * G);
    const int tile_last = cache_start + min((int)blockIdx.x * 64 + 63, R - 1) / G;  // last key of the tile
    const int wave_last = cache_start + min(w0 + 15, R - 1) / G;
    const int nkb = tile_last / KB + 1, b0 = nkb * s / n_splits, b1 = nkb * (s + 1) / n_splits;
    const float* qrow = q + ((size_t)qi * n_heads + h) * D;
    Wave w;
    w.init(qrow, g);
    const float scale = 1.0f / sqrtf((float)D);
    attn_u32x4_t kr[NL], vr[NL];
    auto gload = [&](int b) {
#pragma unroll
        for (int i = 0; i < NL; i++) {
            const int idx = tid + 256 * i;
            const size_t off = ((size_t)min(b * KB + idx / CPR, tile_last) * kv_dim + kv_h * D) * sizeof(CT) + (idx % CPR) * 16;
            kr[i] = *(const attn_u32x4_t*)((const char*)kc + off);
            vr[i] = *(const attn_u32x4_t*)((const char*)vc + off);
        }
    };
    if (b0 < b1) gload(b0);
    for (int b = b0; b < b1; b++) {
        __syncthreads();  // the previous block's reads are done
#pragma unroll
        for (int i = 0; i < NL; i++) {
            const int idx = tid + 256 * i, off = idx / CPR * LD * (int)sizeof(CT) + idx % CPR * 16;
            *(attn_u32x4_t*)((char*)ks + off) = kr[i];
            *(attn_u32x4_t*)((char*)vs + off) = vr[i];
        }
        __syncthreads();
        gload(min(b + 1, b1 - 1));
        if (b * KB > wave_last) continue;  // wave-uniform: every key is behind this wave's rows
        attn_f32x4_t sc[KT];
#pragma unroll
        for (int t = 0; t < KT; t++) {
            attn_u32x4_t k[Wave::NK];
#pragma unroll
            for (int c = 0; c < Wave::NK; c++) k[c] = *(const attn_u32x4_t*)(ks + (t * 16 + r) * LD + Wave::dim0(c, g));
            sc[t] = w.score(k);
        }
        const float a = w.softmax(sc, b * KB, cache_start + qi, scale, g);
        w.pv(sc, a, vs, g, r);
    }
    w.finish();
    const bool live = w0 + r < R;
    const float inv = n_splits > 1 ? 1.0f : 1.0f / w.l;
    // the record, or (one split) the result, of a row
    auto place = [&](int rw) {
        if (n_splits > 1) return part_o + (((size_t)kv_h * R + rw) * n_splits + s) * D;
        return out + ((size_t)(rw / G) * n_heads + kv_h * G + rw % G) * D;
    };
    auto ml = [&](int rw) { return (float2*)(part_ml + 2 * (((size_t)kv_h * R + rw) * n_splits + s)); };
    if (live) {
        float* p = place(row);
#pragma unroll
        for (int t = 0; t < Wave::NDT; t++) *(attn_f32x4_t*)(p + t * 16 + 4 * g) = w.o[t] * inv;
        if (n_splits > 1 && g == 0) *ml(row) = make_float2(w.m, w.l);
    }
    uint64_t todo = __ballot(live && !w.finite());
    todo = (todo | (todo >> 16) | (todo >> 32) | (todo >> 48)) & 0xFFFF;
    for (; todo; todo &= todo - 1) {
        const int rw = w0 + (int)__builtin_ctzll(todo), qx = rw / G;
        const AttnRow x = attn_row_plain<D, CT>(q + ((size_t)qx * n_heads + kv_h * G + rw % G) * D, kc + kv_h * D, vc + kv_h * D,
                                                kv_dim, b0 * KB, min(b1 * KB, cache_start + qx + 1), KB, KB, lane);
        const float xi = n_splits > 1 ? 1.0f : 1.0f / x.l;
        float* p = place(rw);
        if (lane < D / 8) {
#pragma unroll
            for (int i = 0; i < 8; i++) p[lane * 8 + i] = x.acc[i] * xi;
        }
        if (n_splits > 1 && lane == 0) *ml(rw) = make_float2(x.m, x.l);
    }
}

// One wave per row: the splits' records merged in split order.
template <int D>
__global__ __launch_bounds__(256) void attn_rows_merge_kernel(const float* __restrict__ part_o,
                                                              const float* __restrict__ part_ml, int n_splits, int q_len,
                                                              int G, int n_kv_heads, float* __restrict__ out) {
    constexpr int E = D / 64;
    const int R = q_len * G, n_heads = n_kv_heads * G, lane = threadIdx.x & 63;
    const int x = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (x >= R * n_kv_heads) return;  // wave-uniform
    const int kv_h = x / R, rw = x - kv_h * R, qi = rw / G, h = kv_h * G + rw % G;
    const float* po = part_o + (size_t)x * n_splits * D;
    const float* ml = part_ml + (size_t)x * n_splits * 2;
    float M = -INFINITY, L = 0.0f, A[E];
#pragma unroll
    for (int e = 0; e < E; e++) A[e] = 0.0f;
    for (int s = 0; s < n_splits; s++) M = fmaxf(M, ml[2 * s]);
    for (int s = 0; s < n_splits; s++) {
        const float f = ml[2 * s] == -INFINITY ? 0.0f : expf(ml[2 * s] - M);
        L = __builtin_fmaf(f, ml[2 * s + 1], L);
#pragma unroll
        for (int e = 0; e < E; e++) A[e] = __builtin_fmaf(f, po[(size_t)s * D + lane + 64 * e], A[e]);
    }
    const size_t o = ((size_t)qi * n_heads + h) * D;
#pragma unroll
    for (int e = 0; e < E; e++) out[o + lane + 64 * e] = A[e] * (1.0f / L);
}

template <int D, typename CT>
static void launch_attn_rows(const float* q, const void* kc, const void* vc, int cache_start, int q_len, int n_heads,
                             int n_kv_heads, float* out, hipStream_t s, th_device* dev) {
    const int G = n_heads / n_kv_heads, cus = dev->num_cus;
    const size_t R = (size_t)q_len * G, n = (size_t)cache_start + q_len;
    const CT *k = (const CT*)kc, *v = (const CT*)vc;
    // record space: [kv head][row][split] of D sums, then {max, sum}
    auto records = [&](size_t splits, float*& po, float*& pml) {
        const size_t recs = splits > 1 ? R * n_kv_heads * splits : 0;
        po = recs ? (float*)device_scratch(dev, recs * (D + 2) * sizeof(float)) : nullptr;
        pml = po + recs * D;
    };
    float *po, *pml;
    if (R <= 16) {
        // one workgroup per CU at most, each split at least one pass of its waves
        typedef AttnDec<D, CT> T;
        auto decode = [&](auto nw) {
            constexpr int NW = decltype(nw)::value;
            const size_t pass = (size_t)NW * T::KB;
            const size_t per = round_up(std::max(pass, ceil_div(n, (size_t)std::max(1, cus / n_kv_heads))), pass);
            const size_t splits = ceil_div(n, per);
            // (their weights fit the LDS of the waves' rows: at most cus * 16 records of a kv head)
            TH_REQUIRE(splits * R * 8 <= NW * T::REGION, "attention splits exceed the merge's LDS");
            records(splits, po, pml);
            int* counters = device_counters(dev, n_kv_heads);
            auto kern = attn_rows_decode_kernel<D, CT, NW>;
            static std::mutex mu;
            static bool granted = false;
            {
                std::lock_guard<std::mutex> lock(mu);
                if (!granted)
                    TH_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                               (int)(NW * T::REGION)));
                granted = true;
            }
            TH_LAUNCH(kern, dim3((unsigned)n_kv_heads, (unsigned)splits), dim3(64 * NW), NW * T::REGION, s, q, k, v,
                      cache_start, q_len, G, n_kv_heads, (int)per, (int)splits, po, pml, counters, out);
            TH_LAUNCH_CHECK();
        };
        // Up to 2048 keys four waves spread a context over more CUs (1200 keys,
        // D 128: 10.3 against 12.0 us); beyond, eight keep the splits few (8000
        // keys, four query heads on each of 4 kv heads: 15.0 against 20.1).  Two
        // waves a SIMD have too few registers for 256 dims of f32 (9000 keys,
        // four heads on each of 4: 41.9 with four waves, 44.8 with eight).
        if constexpr (D <= 128 || sizeof(CT) == 2) {
            if (n > 2048) {
                decode(std::integral_constant<int, 8>{});
                return;
            }
        }
        decode(std::integral_constant<int, 4>{});
        return;
    }
    const size_t tiles = ceil_div(R, (size_t)64), nkb = ceil_div(n, (size_t)AttnPre<D, CT>::KB);
    // two workgroups per CU, each split at least two key blocks of the longest tile
    const size_t splits = std::max<size_t>(1, std::min({ceil_div((size_t)(2 * cus), tiles * n_kv_heads), nkb / 2, (size_t)16}));
    records(splits, po, pml);
    TH_LAUNCH((attn_rows_kernel<D, CT>), dim3((unsigned)tiles, (unsigned)n_kv_heads, (unsigned)splits), dim3(256), 0, s, q,
              k, v, cache_start, q_len, G, n_kv_heads, (int)splits, po, pml, out);
    TH_LAUNCH_CHECK();
    if (splits > 1) {
        TH_LAUNCH(attn_rows_merge_kernel<D>, dim3((unsigned)ceil_div(R * n_kv_heads, (size_t)4)), dim3(256), 0, s, po, pml,
                  (int)splits, q_len, G, n_kv_heads, out);
        TH_LAUNCH_CHECK();
    }
}

void launch_kv_attention(const float* q, const void* kc, const void* vc, bool f16, size_t cache_start, size_t q_len,
                         size_t n_heads, size_t n_kv_heads, size_t head_dim, float* out, hipStream_t s,
                         th_device* dev) {
    if (q_len == 0 || n_heads == 0) return;
    const bool tuned = head_dim == 64 || head_dim == 128 || head_dim == 256;
    // The split kernel (one workgroup per query, head and 64 keys) remains for
    // what is too small to pay for 16-row tiles.  Its time grows with the work,
    // the tiles' hardly does below a certain size.  Where the lines lie, in us a
    // call (row tiles / split kernel), 8 kv heads unless stated, G query heads each.
    // Up to 16 rows, f16 cache: few keys D 64 128 5.1 / 6.4, D 128 60 5.6 / 6.9,
    // 128 6.5 / 7.0, D 256 60 8.5 / 8.7, 128 11.7 / 8.9; many D 64 G 2 512 8.4 / 7.6,
    // 1024 8.6 / 9.1, G 4 512 8.4 / 7.8, 900 8.6 / 9.8, D 128 G 1 1200 10.0 / 8.4, 2048 10.6 / 10.3, 4000 12.5 / 14.4, G 2
    // 1024 9.9 / 9.7, 8000 16.3 / 35.7, D 256 G 1 4096 19.7 / 17.4, 6144 20.9 / 20.4, G 2
    // 2048 17.9 / 16.6, 3072 18.1 / 22.3.
    // f32 cache (its MFMA has a sixteenth of the rate): few D 64 64 5.2 / 6.3, D 128
    // 32 6.9 / 6.9, 64 7.6 / 7.1, D 256 64 9.1 / 9.0; many D 64 G 1 4096 12.3 / 13.7, G 4
    // 700 9.5 / 8.6, 1024 9.6 / 10.2, D 128 G 1 8192 21.3 / 19.9, 12000 26.8 / 30.9, G 2
    // 3000 16.1 / 19.6, G 4 1200 14.2 / 12.7, D 256 G 1 16000 57.4 / 59.5, G 4 3000 25.2 /
    // 36.7.
    // More rows (queries x keys), f16 cache: D 64 4 kv heads 64 x 256 9.7 / 8.1, 18 x
    // 2000 14.6 / 17.7; D 128 17 x 17 6.4 / 7.4, 30 x 100 9.0 / 8.0, 64 x 128 9.7 / 9.3, 16 kv
    // heads 77 x 80 9.2 / 13.4, 40 x 400 14.8 / 13.0, 100 x 200 12.6 / 14.6; D 256 64 x 128
    // 16.0 / 12.8, 64 x 256 16.8 / 19.1.  f32 cache: D 64 G 2 32 x 512 14.4 / 15.1, 4 kv heads
    // 64 x 256 13.6 / 8.1; D 128 40 x 400 19.1 / 15.7, 100 x 200 17.8 / 18.8; D 256 40 x 140
    // 20.2 / 16.8, 64 x 128 18.3 / 17.7, 64 x 256 20.4 / 29.4.
    const size_t G = n_heads / n_kv_heads, R = q_len * G, n = cache_start + q_len;
    bool tiles;
    const size_t work = q_len * n_heads * n;  // scores
    if (R > 16 && f16) tiles = n <= 64 || work >= (size_t)1 << (n <= 128 && head_dim <= 128 ? 16 : 17);
    else if (R > 16) tiles = work * head_dim >= (size_t)1 << 24;
    else if (f16) tiles = n <= (head_dim <= 128 ? 128 : 64) || n * std::min<size_t>(G, head_dim <= 64 ? 3 : 2) >= (head_dim <= 128 ? 2048 : 6144);
    else if (G > 1) tiles = n <= (head_dim <= 64 ? 64 : 32) || n * std::min<size_t>(G, 4) >= 2048 + 32 * head_dim;
    else tiles = n <= (head_dim <= 64 ? 64 : 32) || n >= (head_dim <= 64 ? 4096 : head_dim <= 128 ? 10240 : 16384);
    if (tuned && !tiles) {
        // enough 64-position chunks per split that the merge fits in LDS
        const size_t max_splits = 64 * 1024 / ((head_dim + 2) * sizeof(float));
        const int subs = (int)std::max<size_t>(1, ceil_div(ceil_div(n, (size_t)ATTN_SUB), max_splits));
        const int n_splits = (int)ceil_div(n, (size_t)subs * ATTN_SUB);
        float* part = (float*)device_scratch(dev, q_len * n_heads * n_splits * (head_dim + 2) * sizeof(float));
        int* counters = device_counters(dev, q_len * n_heads);
        launch_attn_split<false>(q, kc, vc, f16, (int)cache_start, (int)q_len, (int)n_heads, (int)n_kv_heads,
                                 (int)head_dim, subs, n_splits, part, counters, (void*)out, nullptr, s);
        return;
    }
    auto rows = [&](auto d) {
        constexpr int D = decltype(d)::value;
        if (f16)
            launch_attn_rows<D, _Float16>(q, kc, vc, (int)cache_start, (int)q_len, (int)n_heads, (int)n_kv_heads, out, s, dev);
        else
            launch_attn_rows<D, float>(q, kc, vc, (int)cache_start, (int)q_len, (int)n_heads, (int)n_kv_heads, out, s, dev);
    };
    switch (head_dim) {
        case 64: rows(std::integral_constant<int, 64>{}); return;
        case 128: rows(std::integral_constant<int, 128>{}); return;
        case 256: rows(std::integral_constant<int, 256>{}); return;
        default: break;
    }
    TH_REQUIRE(head_dim <= 512, "head_dim above 512 is not supported");
    if (f16)
        TH_LAUNCH(attn_generic_kernel<_Float16>, dim3((unsigned)n_heads, (unsigned)q_len), dim3(64), 0, s, q,
                           (const _Float16*)kc, (const _Float16*)vc, (int)cache_start, (int)n_heads,
                           (int)n_kv_heads, (int)head_dim, out);
    else
        TH_LAUNCH(attn_generic_kernel<float>, dim3((unsigned)n_heads, (unsigned)q_len), dim3(64), 0, s, q,
                           (const float*)kc, (const float*)vc, (int)cache_start, (int)n_heads, (int)n_kv_heads,
                           (int)head_dim, out);
    TH_LAUNCH_CHECK();
}

}  // namespace th

using namespace th;

extern "C" int th_kv_attention(th_device* dev, const th_buffer* q, const th_buffer* k, const th_buffer* v,
                               size_t cache_start, size_t q_len, size_t n_heads, size_t n_kv_heads, size_t head_dim,
                               th_buffer* out) {
    TH_API_BEGIN
    TH_REQUIRE(dev && q && k && v && out, "null argument");
    TH_REQUIRE(n_kv_heads > 0 && n_heads % n_kv_heads == 0, "n_heads must be a multiple of n_kv_heads");
    TH_REQUIRE(k->dtype == v->dtype && (k->dtype == TH_F32 || k->dtype == TH_F16), "caches must both be f32 or f16");
    require_len(q, TH_F32, q_len * n_heads * head_dim, "q");
    require_len(out, TH_F32, q_len * n_heads * head_dim, "out");
    require_len_any(k, (cache_start + q_len) * n_kv_heads * head_dim, "k_cache");
    require_len_any(v, (cache_start + q_len) * n_kv_heads * head_dim, "v_cache");
    launch_kv_attention((const float*)q->ptr, k->ptr, v->ptr, k->dtype == TH_F16, cache_start, q_len, n_heads, n_kv_heads,
                        head_dim, (float*)out->ptr, dev->stream, dev);
    TH_API_END
}
