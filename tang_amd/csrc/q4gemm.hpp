// Launchers of the dense int4 MFMA GEMM (prepared activations) with any
// epilogue: the linear entry points store, the prefill fuses RoPE and SwiGLU.
#pragma once

#include <algorithm>
#include <map>
#include <mutex>

#include "capi_util.hpp"
#include "qlinear.hpp"

namespace th {

// Raise a kernel's dynamic-LDS limit (once per kernel and size).
template <typename K>
inline void set_smem(K kernel, size_t bytes) {
    static std::mutex mu;
    static std::map<const void*, size_t> done;
    if (bytes <= 48 * 1024) return;
    std::lock_guard<std::mutex> lock(mu);
    size_t& d = done[(const void*)kernel];
    if (bytes > d) {
        TH_HIP(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes));
        d = bytes;
    }
}

template <int RT, int CB, int KW, typename ST, typename Epi>
inline void q4_wave_launch(const th_qweight* w, PreparedX xp, size_t m, const Epi& epi, hipStream_t s) {
    auto k = q4_gemm_wave_kernel<RT, CB, KW, ST, Epi>;
    const size_t lds = (size_t)KW * RT * CB * 1024;
    set_smem(k, lds);
    TH_LAUNCH(k, dim3((unsigned)ceil_div(w->Np / 16, (size_t)RT), (unsigned)ceil_div(m, (size_t)(16 * CB))), dim3(64 * KW),
              lds, s, (const uint4*)w->data, (const ST*)w->scales, (const int*)w->row_exp, xp.x, xp.xexp, epi, (int)m,
              (int)w->rows, (int)w->Kp);
    TH_LAUNCH_CHECK();
}

// Weight tiles and waves of a workgroup by the number of workgroups that four
// tiles each would give (`wgs`), per CU: the more there are, the larger the tile
// and the fewer the waves that split its K.  Measured on 256 CUs, us (4x4 / 4x8 / 2x8 / 1x8,
// tiles x waves): 2048 x 2048, m = 512 (256) 15.9 / 15.4 / 18.4 / 21.8; m = 384
// (192) 14.8 / 14.3 / 17.1 / 18.0; m = 192 (96) 13.9 / 12.9 / 11.2 / 13.2;
// m = 64 (32) 13.4 / 11.9 / 10.1 / 9.4; 11008 x 4096, m = 96 (344) 26.2 / 29.4 /
// 30.0 / 38.4.  Up to 32 rows four tiles never pay (22016 x 4096, m = 32: 4x4
// 22.0, 2x4 19.7, 2x8 20.5), and a single block of rows over a long K takes
// sixteen waves (4096 x 11008, m = 16: 1x8 14.8, 1x16 13.3).
template <int CB, typename ST, typename Epi>
inline void q4_wave_shape(const th_qweight* w, PreparedX xp, size_t m, const Epi& epi, hipStream_t s) {
    const size_t wgs = ceil_div(w->Np / 16, (size_t)4) * ceil_div(m, (size_t)(16 * CB)), cus = w->dev->num_cus;
    if constexpr (CB <= 2) {
        if (wgs > cus * 9 / 16) return q4_wave_launch<2, CB, 4, ST>(w, xp, m, epi, s);
    } else {
        if (wgs > cus * 7 / 8) return q4_wave_launch<4, CB, 4, ST>(w, xp, m, epi, s);
        if (wgs > cus * 9 / 16) return q4_wave_launch<4, CB, 8, ST>(w, xp, m, epi, s);
    }
    if (wgs > cus * 9 / 32) return q4_wave_launch<2, CB, 8, ST>(w, xp, m, epi, s);
    if constexpr (CB == 1) {
        if (w->Kp >= 32 * 128) return q4_wave_launch<1, CB, 16, ST>(w, xp, m, epi, s);
    }
    q4_wave_launch<1, CB, 8, ST>(w, xp, m, epi, s);
}

template <int RT, int KW, typename ST, typename Epi>
inline void q4_rows_launch(const th_qweight* w, const float* x, size_t m, size_t ldx, const Epi& epi, hipStream_t s) {
    const size_t lds = (size_t)KW * 4096;
    auto k = q4_gemm_rows_kernel<RT, KW, ST, Epi>;
    set_smem(k, lds);
    TH_LAUNCH(k, dim3((unsigned)ceil_div(w->Np / 16, (size_t)RT)), dim3(64 * KW), lds, s, (const uint4*)w->data,
              (const ST*)w->scales, (const int*)w->row_exp, x, epi, (int)m, (int)w->rows, (int)w->cols, (int)w->Kp,
              (int)ldx);
    TH_LAUNCH_CHECK();
}

// Whether at most 16 rows of f32 go to q4_gemm_rows_kernel unprepared: the
// preparation and its launch (4 to 6 us) against converting all of x again in
// every workgroup.  us, prepared / not, m = 16: 256 x 1024 5.7 / 3.4, 2500 x 2500
// 7.6 / 4.9, 2500 x 6700 11.7 / 9.5, 4096 x 11008 13.0 / 13.7; several workgroups a
// CU: 6700 x 2500 8.3 / 6.3, 11264 x 2048 8.7 / 7.8, 11008 x 4096 12.1 / 12.7.
// Rows that cannot be read in aligned fours are prepared (scalar loads took
// 3333 x 3333 from 76 to 137 us over eight linears).
inline bool q4_rows_direct(const th_qweight* w, const float* x, size_t m, size_t ldx) {
    const size_t tiles = w->Np / 16, cus = w->dev->num_cus;
    return m <= 16 && w->cols % 4 == 0 && ldx % 4 == 0 && ((uintptr_t)x & 15) == 0 &&
           w->cols <= (tiles <= cus ? 8192u : 3072u) && ldx < ((size_t)1 << 25);  // 32-bit offsets into 16 rows
}

// One weight tile a workgroup while that is at most one workgroup a CU, two
// beyond, and four waves instead of eight once there are several (us at m = 16,
// 1x8 / 2x8 / 2x4 tiles x waves: 2048 x 2048 4.4 / 5.1 / 5.4; 5632 x 2048 6.3 /
// 5.2 / 5.5; 11264 x 2048 9.2 / 8.2 / 7.8).
template <typename ST, typename Epi>
inline void q4_gemm_rows(const th_qweight* w, const float* x, size_t m, size_t ldx, const Epi& epi, hipStream_t s) {
    const size_t tiles = w->Np / 16, cus = w->dev->num_cus;
    if (tiles <= cus) q4_rows_launch<1, 8, ST>(w, x, m, ldx, epi, s);
    else if (tiles <= 2 * cus) q4_rows_launch<2, 8, ST>(w, x, m, ldx, epi, s);
    else q4_rows_launch<2, 4, ST>(w, x, m, ldx, epi, s);
}

template <int RT, int CB, typename ST, typename Src = GemmDense, typename Epi>
inline void q4_mfma_launch(const th_qweight* w, PreparedX xp, size_t m, const Epi& epi, hipStream_t s) {
    Src src;
    src.M = (int)m;
    TH_LAUNCH((q4_gemm_mfma_kernel<RT, CB, ST, Src, Epi>),
              dim3((unsigned)ceil_div(w->Np / 16, (size_t)(4 * RT)), (unsigned)ceil_div(m, (size_t)(16 * CB)), 1), dim3(256),
              0, s, (const uint4*)w->data, (const ST*)w->scales, (const int*)w->row_exp, xp.x, xp.xexp, epi, src,
              (int)w->rows, (int)w->Kp, (int)w->Kp);
    TH_LAUNCH_CHECK();
}

// The kernel with activations staged in LDS once a workgroup's waves would
// load them from L2 too often: from some 22 tiles of 64 x 64 a CU (us, wave kernel
// / this one: 22016 x 4096, m = 768 191 / 199, 1024 253 / 249, 1536 381 / 364;
// 11008 x 4096, m = 1536 195 / 220; 4096 x 4096 79 / 102).  128-row blocks
// beyond m = 1024, 64-row ones before.
template <typename ST, typename Epi>
inline void q4_gemm_dense(const th_qweight* w, PreparedX xp, size_t m, const Epi& epi, hipStream_t s) {
    const size_t tiles = ceil_div(w->Np / 16, (size_t)4) * ceil_div(m, (size_t)64);
    if (tiles >= (size_t)w->dev->num_cus * 175 / 8) {
        if (m > 1024) q4_mfma_launch<2, 8, ST>(w, xp, m, epi, s);
        else q4_mfma_launch<2, 4, ST>(w, xp, m, epi, s);
        return;
    }
    if (m <= 16) q4_wave_shape<1, ST>(w, xp, m, epi, s);
    else if (m <= 32) q4_wave_shape<2, ST>(w, xp, m, epi, s);
    else if (m <= 48) q4_wave_shape<3, ST>(w, xp, m, epi, s);
    else q4_wave_shape<4, ST>(w, xp, m, epi, s);
}

}  // namespace th
