// Launchers and C entry points for the quantized linear kernels.
#include <cstdlib>

#include "aql.hpp"
#include "capi_util.hpp"
#include "q4gemm.hpp"
#include "q8gemm.hpp"
#include "qlinear.hpp"

namespace th {

// Whether a q8 linear runs as GEMV launches of four rows: up to four rows,
// and up to eight on a matrix of at most 4M weights, where two launches cost
// no more than the MFMA GEMM and its split-K reduction (2048 x 2048, m = 5:
// 8.5 against 9.1 us).  Beyond that the GEMM reads the weights once where the
// GEMV took a launch per four rows: 11008 x 4096, f32 rows, m = 5 28.0 -> 16
// us, m = 100 429 -> 51 us; at four rows on 4096 x 4096 the GEMV is still the
// faster one (7.9 against 12 us).
static bool q8_uses_gemv(const th_qweight* w, size_t m) {
    return m <= 4 || (m <= 8 && w->rows * w->cols <= ((size_t)1 << 22));
}

// Vector activation loads need K, the row stride and the base 16-byte aligned.
static bool x_vec_ok(const void* x, size_t ldx, size_t K) {
    return K % 8 == 0 && ldx % 8 == 0 && ((uintptr_t)x & 15) == 0;
}

template <int M, bool XF32, typename ST, bool VEC, typename Src>
static void q4_gemv_launch_v(const th_qweight* w, const void* x, size_t ldx, float* y, size_t ldy, hipStream_t s,
                             Src src) {
    constexpr int MR = XF32 ? 2 * M : M;
    EpiStore epi{y, (int)ldy};
    if (M == 1 && w->Np / 16 < 512 && w->Kp / 128 >= 64) {  // few tiles, long K: sixteen waves per tile
        const size_t smem = Q4GemvSmem<MR, 16>::bytes((int)(w->Kp / 128));
        TH_REQUIRE(smem <= 160 * 1024, "activation too large for the LDS-staged GEMV");
        auto k = q4_gemv_kernel<MR, XF32, VEC, ST, EpiStore, 2, 4, 16, false, Src>;
        set_smem(k, smem);
        TH_LAUNCH(k, dim3((unsigned)(w->Np / 16)), dim3(1024), smem, s, (const uint4*)w->data,
                           (const ST*)w->scales, x, (int)w->cols, (int)w->Kp, (int)w->rows, (int)ldx, epi, NormArgs{}, src);
    } else if (MR >= 3 || w->Np / 16 < 512) {  // few tiles, or 3+ staged rows: split K over eight waves per tile
        const size_t smem = Q4GemvSmem<MR, 8>::bytes((int)(w->Kp / 128));
        TH_REQUIRE(smem <= 160 * 1024, "activation too large for the LDS-staged GEMV");
        auto k = q4_gemv_kernel<MR, XF32, VEC, ST, EpiStore, 2, 4, 8, false, Src>;
        set_smem(k, smem);
        TH_LAUNCH(k, dim3((unsigned)(w->Np / 16)), dim3(512), smem, s, (const uint4*)w->data,
                           (const ST*)w->scales, x, (int)w->cols, (int)w->Kp, (int)w->rows, (int)ldx, epi, NormArgs{}, src);
    } else {
        const size_t smem = Q4GemvSmem<MR, 4>::bytes((int)(w->Kp / 128));
        TH_REQUIRE(smem <= 160 * 1024, "activation too large for the LDS-staged GEMV");
        auto k = q4_gemv_kernel<MR, XF32, VEC, ST, EpiStore, 2, 4, 4, false, Src>;
        set_smem(k, smem);
        TH_LAUNCH(k, dim3((unsigned)(w->Np / 16)), dim3(256), smem, s, (const uint4*)w->data,
                           (const ST*)w->scales, x, (int)w->cols, (int)w->Kp, (int)w->rows, (int)ldx, epi, NormArgs{}, src);
    }
    TH_LAUNCH_CHECK();
}

template <int M, bool XF32, typename ST, typename Src = SingleMatrix>
static void q4_gemv_launch(const th_qweight* w, const void* x, size_t ldx, float* y, size_t ldy, hipStream_t s,
                           Src src = Src{}) {
    if (x_vec_ok(x, ldx, w->cols)) q4_gemv_launch_v<M, XF32, ST, true>(w, x, ldx, y, ldy, s, src);
    else q4_gemv_launch_v<M, XF32, ST, false>(w, x, ldx, y, ldy, s, src);
}

template <bool XF32, typename ST>
static void q4_gemv_dispatch(const th_qweight* w, const void* x, size_t m, size_t ldx, float* y,
                             size_t ldy, hipStream_t s) {
    switch (m) {
        case 1: q4_gemv_launch<1, XF32, ST>(w, x, ldx, y, ldy, s); break;
        case 2: q4_gemv_launch<2, XF32, ST>(w, x, ldx, y, ldy, s); break;
        default: throw Error(TH_ERR_INVALID, "q4 gemv: m out of range");
    }
}

// M block rows (4, 8 or 16; twice that staged after f32 hi/lo splitting), m
// of them live: NW waves split K, and each workgroup takes ceil(tiles / CUs)
// consecutive tiles so that the whole grid is resident at once and the
// staged activations are read once per workgroup.
template <int M, bool XF32, typename ST, bool VEC, bool RT>
static void q4_span_launch_v(const th_qweight* w, const void* x, size_t m, size_t ldx, float* y, size_t ldy,
                             hipStream_t s, int cus) {
    constexpr int MR = XF32 ? 2 * M : M;
    constexpr int NW = MR >= 16 ? 16 : 8, WPE = MR >= 16 ? 1 : 4;
    using Src = SingleMatrixSpan<RT>;
    const int tiles = (int)(w->Np / 16);
    Src src;
    src.tiles = tiles;
    src.per = (int)ceil_div((size_t)tiles, (size_t)cus);
    src.rows = (int)m;
    const unsigned grid = (unsigned)ceil_div((size_t)tiles, (size_t)src.per);
    const int GQ = (int)(w->Kp / 128);
    size_t smem = Q4GemvSmem<MR, NW>::bytes(GQ);
    auto k = q4_gemv_kernel<MR, XF32, VEC, ST, EpiStore, 2, WPE, NW, false, Src>;
    // two or three tiles per workgroup: streamed side by side (one reduction)
    if (src.per == 2) {
        k = q4_gemv_kernel<MR, XF32, VEC, ST, EpiStore, 2, WPE, NW, false, Src, 2>;
        smem = Q4GemvSmem<MR, NW, 2>::bytes(GQ);
    } else if (src.per == 3) {
        k = q4_gemv_kernel<MR, XF32, VEC, ST, EpiStore, 2, WPE, NW, false, Src, 3>;
        smem = Q4GemvSmem<MR, NW, 3>::bytes(GQ);
    }
    TH_REQUIRE(smem <= 160 * 1024, "activation too large for the LDS-staged GEMV");
    set_smem(k, smem);
    TH_LAUNCH(k, dim3(grid), dim3(64 * NW), smem, s, (const uint4*)w->data, (const ST*)w->scales, x,
                       (int)w->cols, (int)w->Kp, (int)w->rows, (int)ldx, EpiStore{y, (int)ldy}, NormArgs{}, src);
    TH_LAUNCH_CHECK();
}

template <int M, bool XF32, typename ST>
static void q4_span_launch(const th_qweight* w, const void* x, size_t m, size_t ldx, float* y, size_t ldy,
                           hipStream_t s, int cus) {
    const bool vec = x_vec_ok(x, ldx, w->cols);
    if (m == M) {  // all rows live: constant-folded staging
        if (vec) q4_span_launch_v<M, XF32, ST, true, false>(w, x, m, ldx, y, ldy, s, cus);
        else q4_span_launch_v<M, XF32, ST, false, false>(w, x, m, ldx, y, ldy, s, cus);
    } else {
        if (vec) q4_span_launch_v<M, XF32, ST, true, true>(w, x, m, ldx, y, ldy, s, cus);
        else q4_span_launch_v<M, XF32, ST, false, true>(w, x, m, ldx, y, ldy, s, cus);
    }
}

// Sum KS split-K partials [KS][m][N] in split order (then add it to y when
// add is set: the fused residual add).  VEC4: four consecutive columns per
// thread with 16-byte accesses (N and ldy multiples of 4); same sums.
template <bool VEC4>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ part, float* __restrict__ y,
                                                            int M, int N, int ldy, int KS, int add) {
    if (VEC4) {
        const int N4 = N >> 2;
        const int total = M * N4;
        for (int i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
            const int m = i / N4, n = (i - m * N4) * 4;
            float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            for (int s = 0; s < KS; s++) {
                const float4 p = *(const float4*)(part + ((size_t)s * M + m) * N + n);
                v.x += p.x; v.y += p.y; v.z += p.z; v.w += p.w;
            }
            float4* yp = (float4*)(y + (size_t)m * ldy + n);
            if (add) {
                const float4 o = *yp;
                v = make_float4(o.x + v.x, o.y + v.y, o.z + v.z, o.w + v.w);
            }
            *yp = v;
        }
        return;
    }
    const size_t total = (size_t)M * N;
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const size_t m = i / N, n = i - m * N;
        float v = 0.0f;
        for (int s = 0; s < KS; s++) v += part[((size_t)s * M + m) * N + n];
        y[m * ldy + n] = add ? y[m * ldy + n] + v : v;
    }
}

void launch_splitk_reduce(const float* part, float* y, size_t m, size_t n, size_t ldy, size_t ks, bool add,
                          hipStream_t s) {
    const size_t total = m * n;
    const bool vec4 = n % 4 == 0 && ldy % 4 == 0 && ((uintptr_t)y & 15) == 0 && total < (1u << 31);
    if (vec4)
        TH_LAUNCH(splitk_reduce_kernel<true>, dim3((unsigned)std::min<size_t>(ceil_div(total / 4, 256), 4096)),
                  dim3(256), 0, s, part, y, (int)m, (int)n, (int)ldy, (int)ks, (int)add);
    else
        TH_LAUNCH(splitk_reduce_kernel<false>, dim3((unsigned)std::min<size_t>(ceil_div(total, 256), 4096)), dim3(256),
                  0, s, part, y, (int)m, (int)n, (int)ldy, (int)ks, (int)add);
    TH_LAUNCH_CHECK();
}

// Convert m activation rows (f32 or bf16, rows of ldx) into the MFMA GEMM's
// prepared layout in the device's operand workspace.
static size_t prepared_rows_bytes(size_t m, size_t Kp, bool blocked) {
    return blocked ? round_up(m, 16) * Kp * 2 : round_up(m * Kp * 2, 256);
}
size_t prepared_x_bytes(size_t m, size_t Kp, bool blocked) {
    return prepared_rows_bytes(m, Kp, blocked) + round_up(m * sizeof(int), 256);
}

PreparedX prepare_x(th_device* dev, const void* x, bool xf32, size_t m, size_t ldx, size_t K, size_t Kp,
                    hipStream_t s, const int* rows, void* workspace, bool blocked) {
    TH_REQUIRE(m * Kp * 2 < 0x7FFFFFF0u, "prepared activations above 2 GiB");  // 32-bit buffer offsets
    const size_t xbytes = prepared_rows_bytes(m, Kp, blocked);
    char* ws = workspace ? (char*)workspace : (char*)device_scratch_x(dev, prepared_x_bytes(m, Kp, blocked));
    PreparedX p{(const uint16_t*)ws, (const int*)(ws + xbytes)};
    const size_t cpr = Kp / 8;
    if (cpr <= 8 * 256) {  // row per workgroup, in registers
        auto row_kernel = [&](auto xf, auto u) {
            constexpr bool XF = decltype(xf)::value;
            constexpr int UU = decltype(u)::value;
            TH_LAUNCH((q4_gemm_xprep_row_kernel<XF, UU>), dim3((unsigned)m), dim3(256), 0, s, x, (int)ldx, (int)K,
                      (int)Kp, (int)blocked, rows, (uint4*)ws, (int*)(ws + xbytes));
        };
        auto by_u = [&](auto xf) {
            if (cpr <= 256) row_kernel(xf, std::integral_constant<int, 1>{});
            else if (cpr <= 512) row_kernel(xf, std::integral_constant<int, 2>{});
            else if (cpr <= 1024) row_kernel(xf, std::integral_constant<int, 4>{});
            else row_kernel(xf, std::integral_constant<int, 8>{});
        };
        if (xf32) by_u(std::true_type{});
        else by_u(std::false_type{});
        TH_LAUNCH_CHECK();
        return p;
    }
    const unsigned grid = (unsigned)ceil_div(m, (size_t)4);
    if (xf32)
        TH_LAUNCH((q4_gemm_xprep_kernel<true>), dim3(grid), dim3(256), 0, s, x, (int)ldx, (int)K, (int)Kp,
                           (int)m, (int)blocked, rows, (uint4*)ws, (int*)(ws + xbytes));
    else
        TH_LAUNCH((q4_gemm_xprep_kernel<false>), dim3(grid), dim3(256), 0, s, x, (int)ldx, (int)K, (int)Kp,
                           (int)m, (int)blocked, rows, (uint4*)ws, (int*)(ws + xbytes));
    TH_LAUNCH_CHECK();
    return p;
}

static EpiGemmStore q4_store_epi(const th_qweight* w, float* y, size_t ldy, bool accumulate) {
    return {y, (int)ldy, (int)accumulate, w->rows % 4 == 0 && ldy % 4 == 0 && ((uintptr_t)y & 15) == 0};
}

template <typename ST>
static void q4_gemm_store(const th_qweight* w, PreparedX xp, size_t m, float* y, size_t ldy, hipStream_t s,
                          bool accumulate) {
    q4_gemm_dense<ST>(w, xp, m, q4_store_epi(w, y, ldy, accumulate), s);
}

// ws (optional, ws_bytes long): the caller's workspace for the MFMA path's
// prepared activations.
template <bool XF32, typename ST>
static void q4_linear_t(const th_qweight* w, const void* x, size_t m, size_t ldx, float* y, size_t ldy,
                        hipStream_t s, th_device* dev, void* ws = nullptr, size_t ws_bytes = 0) {
    const int GQ = (int)(w->Kp / 128), cus = dev && dev->num_cus > 0 ? dev->num_cus : 256;
    // staged rows fit LDS (with the side-by-side tiles' extra, the largest case)
    const bool fits8 = Q4GemvSmem<8, 8, 3>::bytes(GQ) <= 160 * 1024;
    const bool fits16 = Q4GemvSmem<16, 16, 3>::bytes(GQ) <= 160 * 1024;
    const bool fits4 = Q4GemvSmem<XF32 ? 8 : 4, 8, 3>::bytes(GQ) <= 160 * 1024;
    // m <= 2: one tile per workgroup; 3..16: a 4-, 8- or 16-row block staged
    // once per workgroup over ceil(tiles / CUs) tiles (config 2, M=4: 8.3 ->
    // 7.6 us; M=1 is faster with one tile per workgroup, 6.7 against 7.0)
    if (m <= 2 && fits4) q4_gemv_dispatch<XF32, ST>(w, x, m, ldx, y, ldy, s);
    else if (m <= 4 && fits4) q4_span_launch<4, XF32, ST>(w, x, m, ldx, y, ldy, s, cus);
    else if (XF32 && m <= 8 && fits16) q4_span_launch<8, true, ST>(w, x, m, ldx, y, ldy, s, cus);
    else if (!XF32 && m <= 8 && fits8) q4_span_launch<8, false, ST>(w, x, m, ldx, y, ldy, s, cus);
    else if (!XF32 && m <= 16 && fits16) q4_span_launch<16, false, ST>(w, x, m, ldx, y, ldy, s, cus);
    else {  // activations prepared once per call, then the MFMA GEMM
        // the whole blocks' padding rows go into the workspace's slack
        if (ws)
            TH_REQUIRE(prepared_x_bytes(m, w->Kp, false) <= TH_NOALLOC_SCRATCH_BYTES,
                       "workspace too small for the prepared activations (m x K too large)");
        if constexpr (XF32) {
            if (q4_rows_direct(w, (const float*)x, m, ldx)) {
                q4_gemm_rows<ST>(w, (const float*)x, m, ldx, q4_store_epi(w, y, ldy, false), s);
                return;
            }
        }
        const bool blocked = !ws || prepared_x_bytes(m, w->Kp) <= ws_bytes;
        const PreparedX xp = prepare_x(dev, x, XF32, m, ldx, w->cols, w->Kp, s, nullptr, ws, blocked);
        if (blocked) q4_gemm_store<ST>(w, xp, m, y, ldy, s, false);
        else q4_mfma_launch<2, 4, ST, GemmDenseRows>(w, xp, m, q4_store_epi(w, y, ldy, false), s);
    }
}

void launch_q4_linear_prepared(const th_qweight* w, PreparedX xp, size_t m, float* y, size_t ldy, hipStream_t s,
                               bool accumulate) {
    TH_REQUIRE(w && w->bits == 4, "not a q4 weight");
    if (m == 0) return;
    if (w->scale_dtype == TH_F16) q4_gemm_store<_Float16>(w, xp, m, y, ldy, s, accumulate);
    else q4_gemm_store<float>(w, xp, m, y, ldy, s, accumulate);
}

void launch_q4_linear(const th_qweight* w, const void* x, th_dtype xdt, size_t m, size_t ldx, float* y,
                      size_t ldy, hipStream_t s, th_device* dev, void* ws, size_t ws_bytes) {
    TH_REQUIRE(w && w->bits == 4, "not a q4 weight");
    TH_REQUIRE(xdt == TH_F32 || xdt == TH_BF16, "activations must be f32 or bf16");
    if (m == 0) return;
    const bool f32 = xdt == TH_F32;
    if (w->scale_dtype == TH_F16) {
        if (f32) q4_linear_t<true, _Float16>(w, x, m, ldx, y, ldy, s, dev, ws, ws_bytes);
        else q4_linear_t<false, _Float16>(w, x, m, ldx, y, ldy, s, dev, ws, ws_bytes);
    } else {
        if (f32) q4_linear_t<true, float>(w, x, m, ldx, y, ldy, s, dev, ws, ws_bytes);
        else q4_linear_t<false, float>(w, x, m, ldx, y, ldy, s, dev, ws, ws_bytes);
    }
}

template <int M, bool XF32, bool PR, bool VEC>
static void q8_launch_v(const th_qweight* w, const void* x, size_t ldx, float* y, size_t ldy, hipStream_t s) {
    // eight waves split each tile's K (config 1: 5.33 us; four waves 5.88,
    // sixteen 6.2-6.3; 2, 6 or 8 chunks in flight per wave instead of 4 were
    // slower)
    constexpr int NW = 8;
    const size_t smem = Q8GemvSmem<M, NW>::bytes((int)w->Kp);
    TH_REQUIRE(smem <= 160 * 1024, "activation too large for the LDS-staged GEMV");
    auto k = q8_gemv_kernel<M, XF32, VEC, PR, EpiStore, NW>;
    set_smem(k, smem);
    EpiStore epi{y, (int)ldy};
    TH_LAUNCH(k, dim3((unsigned)(w->Np / 16)), dim3(64 * NW), smem, s, (const uint4*)w->data,
                       (const float*)w->scales, x, (int)w->cols, (int)w->Kp, (int)w->rows, (int)ldx, epi);
    TH_LAUNCH_CHECK();
}

template <int M, bool XF32, bool PR>
static void q8_launch(const th_qweight* w, const void* x, size_t ldx, float* y, size_t ldy, hipStream_t s) {
    if (x_vec_ok(x, ldx, w->cols)) q8_launch_v<M, XF32, PR, true>(w, x, ldx, y, ldy, s);
    else q8_launch_v<M, XF32, PR, false>(w, x, ldx, y, ldy, s);
}

// K splits of the q8 GEMM: `base` workgroups times ks, chosen so that the
// busiest CU has little more work than the average one, and two workgroups to
// overlap where the work allows (alone on its CU a workgroup waits for each
// step's loads).  11008 x 4096 at m = 100 (172 workgroups) runs in 74 us
// unsplit, 45.9 with 2 splits, 37.0 with 4, 44.3 with 5; 4096 x 4096 at m = 100
// (64) in 21.2 with 8 and 23.8 with 12.  Each split keeps four 64-wide chunks.
static size_t q8_gemm_splits(size_t base, size_t NCH, size_t cus) {
    size_t best = 1;
    double best_fill = 0.0;
    for (size_t ks = 1; ks <= std::min<size_t>(16, std::max<size_t>(1, NCH / 4)); ks++) {
        if (ks > 1 && base * ks > 3 * cus) break;
        const size_t per_cu = ceil_div(base * ks, cus);
        const double fill = (double)(base * ks) / (double)(per_cu * cus) * (per_cu == 1 ? 0.7 : 1.0);
        if (fill > best_fill) { best_fill = fill; best = ks; }
    }
    return best;
}

template <int RT, int CB, int KG, bool XF32, bool PR, bool VEC>
static void q8_gemm_launch(const th_qweight* w, const void* x, size_t m, size_t ldx, float* y, size_t ldy,
                           hipStream_t s, th_device* dev) {
    const size_t NT = w->Np / 16, NCH = w->Kp / 64;
    const unsigned gx = (unsigned)ceil_div(NT, (size_t)(4 * RT)), gy = (unsigned)ceil_div(m, (size_t)(16 * CB));
    const size_t part = m * w->rows * sizeof(float);
    size_t ks = workspace_splits(dev, q8_gemm_splits((size_t)gx * gy, NCH, (size_t)dev->num_cus), part, s);
    const size_t cps = round_up(ceil_div(NCH, ks), (size_t)KG);
    ks = ceil_div(NCH, cps);
    float* out = ks > 1 ? (float*)device_scratch(dev, ks * part) : y;
    const int ldo = ks > 1 ? (int)w->rows : (int)ldy;
    TH_LAUNCH((q8_gemm_kernel<RT, CB, KG, XF32, VEC, PR>), dim3(gx, gy, (unsigned)ks), dim3(256), 0, s,
              (const uint4*)w->data, (const float*)w->scales, x, out, (int)m, (int)w->rows, (int)w->cols, (int)w->Kp,
              (int)ldx, ldo, m * w->rows, (int)cps);
    TH_LAUNCH_CHECK();
    if (ks > 1) launch_splitk_reduce(out, y, m, w->rows, ldy, ks, false, s);
}

template <bool XF32, bool PR, bool VEC>
static void q8_gemm_dispatch(const th_qweight* w, const void* x, size_t m, size_t ldx, float* y, size_t ldy,
                             hipStream_t s, th_device* dev) {
    if (m <= 16) q8_gemm_launch<2, 1, 2, XF32, PR, VEC>(w, x, m, ldx, y, ldy, s, dev);
    else if (m <= 32) q8_gemm_launch<2, 2, XF32 && !PR ? 1 : 2, XF32, PR, VEC>(w, x, m, ldx, y, ldy, s, dev);
    else q8_gemm_launch<2, 4, XF32 ? 1 : 2, XF32, PR, VEC>(w, x, m, ldx, y, ldy, s, dev);
}

template <bool XF32, bool PR>
static void q8_dispatch(const th_qweight* w, const void* x, size_t m, size_t ldx, float* y, size_t ldy,
                        hipStream_t s, th_device* dev) {
    if (!q8_uses_gemv(w, m)) {
        // the rows that the GEMV stages bound K for every m above three
        TH_REQUIRE((Q8GemvSmem<4, 8>::bytes((int)w->Kp)) <= 160 * 1024, "activation too large for the LDS-staged GEMV");
        constexpr size_t ROWS = (size_t)1 << 21;  // a grid has at most 65535 blocks of 64 rows
        for (size_t m0 = 0; m0 < m; m0 += ROWS) {
            const void* xo = (const char*)x + m0 * ldx * (XF32 ? 4 : 2);
            float* yo = y + m0 * ldy;
            const size_t mm = std::min(ROWS, m - m0);
            if (x_vec_ok(xo, ldx, w->cols)) q8_gemm_dispatch<XF32, PR, true>(w, xo, mm, ldx, yo, ldy, s, dev);
            else q8_gemm_dispatch<XF32, PR, false>(w, xo, mm, ldx, yo, ldy, s, dev);
        }
        return;
    }
    for (size_t m0 = 0; m0 < m; m0 += 4) {
        const void* xo = (const char*)x + m0 * ldx * (XF32 ? 4 : 2);
        float* yo = y + m0 * ldy;
        switch (std::min<size_t>(4, m - m0)) {
            case 1: q8_launch<1, XF32, PR>(w, xo, ldx, yo, ldy, s); break;
            case 2: q8_launch<2, XF32, PR>(w, xo, ldx, yo, ldy, s); break;
            case 3: q8_launch<3, XF32, PR>(w, xo, ldx, yo, ldy, s); break;
            default: q8_launch<4, XF32, PR>(w, xo, ldx, yo, ldy, s); break;
        }
    }
}

void launch_q8_linear(const th_qweight* w, const void* x, th_dtype xdt, size_t m, size_t ldx, float* y,
                      size_t ldy, hipStream_t s, th_device* dev) {
    TH_REQUIRE(w && w->bits == 8, "not a q8 weight");
    TH_REQUIRE(xdt == TH_F32 || xdt == TH_BF16, "activations must be f32 or bf16");
    if (m == 0) return;
    if (xdt == TH_F32) {
        if (w->per_row) q8_dispatch<true, true>(w, x, m, ldx, y, ldy, s, dev);
        else q8_dispatch<true, false>(w, x, m, ldx, y, ldy, s, dev);
    } else {
        if (w->per_row) q8_dispatch<false, true>(w, x, m, ldx, y, ldy, s, dev);
        else q8_dispatch<false, false>(w, x, m, ldx, y, ldy, s, dev);
    }
}

}  // namespace th

using namespace th;

extern "C" {

int th_gemm_q4(th_device* dev, const th_buffer* x, size_t m, const th_qweight* w, th_buffer* y) {
    TH_API_BEGIN
    TH_REQUIRE(dev && x && w && y, "null argument");
    TH_REQUIRE(w->bits == 4, "weight is not q4");
    require_len_any(x, m * w->cols, "x");
    require_len(y, TH_F32, m * w->rows, "y");
    launch_q4_linear(w, x->ptr, x->dtype, m, w->cols, (float*)y->ptr, w->rows, dev->stream, dev);
    TH_API_END
}

int th_gemm_q4_noalloc(th_device* dev, const th_buffer* x, size_t m, const th_qweight* w, th_buffer* y) {
    TH_API_BEGIN
    TH_REQUIRE(dev && x && w && y, "null argument");
    TH_REQUIRE(w->bits == 4, "weight is not q4");
    TH_REQUIRE(dev->noalloc_scratch, "no workspace address for this device");
    require_len_any(x, m * w->cols, "x");
    require_len(y, TH_F32, m * w->rows, "y");
    launch_q4_linear(w, x->ptr, x->dtype, m, w->cols, (float*)y->ptr, w->rows, dev->stream, dev, dev->noalloc_scratch,
                     TH_NOALLOC_SCRATCH_BYTES + NOALLOC_SLACK);
    TH_API_END
}

int th_gemv_q8(th_device* dev, const th_buffer* x, size_t m, const th_qweight* w, th_buffer* y) {
    TH_API_BEGIN
    TH_REQUIRE(dev && x && w && y, "null argument");
    TH_REQUIRE(w->bits == 8, "weight is not q8");
    require_len_any(x, m * w->cols, "x");
    require_len(y, TH_F32, m * w->rows, "y");
    launch_q8_linear(w, x->ptr, x->dtype, m, w->cols, (float*)y->ptr, w->rows, dev->stream, dev);
    TH_API_END
}

int th_bench_linear(th_device* dev, const th_buffer* x, size_t m, th_qweight* const* ws, size_t n_w, th_buffer* y,
                    size_t iters, int use_graph, float* ms) {
    TH_API_BEGIN
    TH_REQUIRE(dev && x && ws && n_w > 0 && y && ms, "null argument");
    const th_qweight* w0 = ws[0];
    for (size_t i = 0; i < n_w; i++)
        TH_REQUIRE(ws[i] && ws[i]->bits == w0->bits && ws[i]->rows == w0->rows && ws[i]->cols == w0->cols,
                   "weights must share one shape");
    require_len_any(x, m * w0->cols, "x");
    require_len(y, TH_F32, m * w0->rows, "y");
    auto call = [&](size_t i) {
        const th_qweight* w = ws[i % n_w];
        if (w->bits == 4) launch_q4_linear(w, x->ptr, x->dtype, m, w->cols, (float*)y->ptr, w->rows, dev->stream, dev);
        else launch_q8_linear(w, x->ptr, x->dtype, m, w->cols, (float*)y->ptr, w->rows, dev->stream, dev);
    };
    call(0);  // sizes the workspace before any capture
    TH_HIP(hipStreamSynchronize(dev->stream));
    if (use_graph == 2) {
        // The GEMVs store their output write-through: no release fences
        // between the launches.
        const bool wt = w0->bits == 8 ? q8_uses_gemv(w0, m) : m <= 16;
        // Every call reads x and its weights and writes y: no call reads what
        // another writes (independent).
        // One sequence: whole passes over the copies (at least 240 launches,
        // so the timed launches run in the steady state of a busy queue and
        // every copy was last read n_w launches earlier), two clock stamps
        // back to back (the span of a stamp kernel and its dispatch), one
        // more pass, a clock stamp, the `iters` timed launches from copy 0,
        // a last stamp.  The time is the last interval less the stamps' own
        // span.  The sequence's system-scope acquire and release sit on its
        // first and last packets, outside both intervals.  It is replayed
        // twice; the second replay is timed.
        const size_t pre = ceil_div(std::max<size_t>(240, n_w), n_w) * n_w;
        AqlSeq* seq = aql_record(dev, wt, [&] {
            for (size_t i = 0; i < pre; i++) call(i);
            aql_stamp_launch(dev, 2);
            aql_stamp_launch(dev, 3);
            for (size_t i = 0; i < n_w; i++) call(i);
            aql_stamp_launch(dev, 0);
            for (size_t i = 0; i < iters; i++) call(i);
            aql_stamp_launch(dev, 1);
        }, true);
        try {
            aql_submit(*seq);  // warm replay
            aql_wait(dev);
            aql_submit(*seq);
            *ms = aql_stamped_ms(dev) - aql_stamp_span_ms(dev);
        } catch (...) {
            aql_free(seq);
            throw;
        }
        aql_free(seq);
    } else if (use_graph) {
        hipGraph_t g;
        hipGraphExec_t ge;
        TH_HIP(hipStreamBeginCapture(dev->stream, hipStreamCaptureModeThreadLocal));
        for (size_t i = 0; i < iters; i++) call(i);
        TH_HIP(hipStreamEndCapture(dev->stream, &g));
        TH_HIP(hipGraphInstantiate(&ge, g, nullptr, nullptr, 0));
        TH_HIP(hipGraphLaunch(ge, dev->stream));  // warm replay
        // then one stream-launched pass over the copies in cycle order, so
        // that the timed replay continues the cycle: every launch's weights
        // were last read n_w launches earlier (beyond the last-level cache
        // when n_w copies exceed it), whatever the number of launches
        for (size_t i = 0; i < n_w; i++) call(i);
        TH_HIP(hipEventRecord(dev->ev_start, dev->stream));
        TH_HIP(hipGraphLaunch(ge, dev->stream));
        TH_HIP(hipEventRecord(dev->ev_stop, dev->stream));
        TH_HIP(hipEventSynchronize(dev->ev_stop));
        TH_HIP(hipGraphExecDestroy(ge));
        TH_HIP(hipGraphDestroy(g));
    } else {
        for (size_t i = 0; i < n_w; i++) call(i);
        TH_HIP(hipEventRecord(dev->ev_start, dev->stream));
        for (size_t i = 0; i < iters; i++) call(i);
        TH_HIP(hipEventRecord(dev->ev_stop, dev->stream));
        TH_HIP(hipEventSynchronize(dev->ev_stop));
    }
    if (use_graph != 2) TH_HIP(hipEventElapsedTime(ms, dev->ev_start, dev->ev_stop));
    TH_API_END
}

}  // extern "C"
