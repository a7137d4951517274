// What the two halves of the purified-Born dispatch (purified_fwd.hip,
// purified_bwd.hip: one translation unit each, they take minutes to compile)
// share: which kernels take which problems.
#pragma once

#include "born_f32.h"
#include "purified.h"

namespace qdl {

inline int purified_padded_dim(int D) { return D <= 32 ? 32 : D <= 64 ? 64 : D <= 128 ? 128 : 256; }

// 16-bit inputs with document ids at head dims below 128 other than 64 (or
// with a window without causality): the generic 16-bit-MFMA kernels'
// purified mode (purified_wide.hip).
hipError_t purified_wide_fwd_launch(int dtype, const PurArgs& a, hipStream_t s);
hipError_t purified_wide_bwd_launch(int dtype, const PurArgs& a, hipStream_t s);
// 128 < D <= 256 (documents with a causal window or none): the wide-row
// DMA-ring kernels' purified mode (born_fwd_d256.hip, born_bwd_d256.hip).
hipError_t purified_fwd_d256_launch(int dtype, const PurArgs& a, hipStream_t s);
hipError_t purified_bwd_d256_launch(int dtype, const PurArgs& a, hipStream_t s);

// Whether a call may take the wave-split kernels (born_f32.h, born_split16.h).
// Where scale or tau is trained in fp32 or fp16 it keeps the other kernels:
// dscale is a cancelling sum, which another summation order in the output (its
// last bits) moves by up to 1e-3 (fp32) and 4e-3 (fp16), no nearer to or
// further from float64 (1e-3 and 4e-2 off either way).
template <class IN>
inline bool purified_split_ok(const PurArgs& a) {
    return std::is_same<IN, BF16>::value || !a.param_grads;
}

// fp32 inputs up to D = 128 but for f32_staged (born_fwd_f32.hip, born_bwd_f32.hip).
hipError_t purified_fwd_f32_launch(const PurArgs& a, hipStream_t s);
hipError_t purified_bwd_f32_launch(const PurArgs& a, hipStream_t s);

// The bf16-MFMA kernels address one (batch, head) slice with 32-bit buffer
// offsets (rows up to T + 256 of 2 D bytes); longer slices take the generic
// kernels, as the Born dispatch does.
// Sliding windows: without documents any window (kWindow causal, kWindowNC
// not); with documents a causal one (the wavelet models' purified layers run
// causal with a window and document ids).
inline bool purified_window_ok(const PurArgs& a) { return a.window == 0 || a.is_causal; }

inline bool purified_fast_ok(const PurArgs& a) {
    return a.D == 64 && a.doc == nullptr && ((int64_t)a.T + 256) * a.D * 2 < ((int64_t)1 << 31);
}

// D < 64 (a multiple of 8) on the D = 64 kernels with the columns past D zero.
inline bool purified_narrow_ok(const PurArgs& a) {
    return a.D < 64 && a.doc == nullptr && ((int64_t)a.T + 256) * 64 * 2 < ((int64_t)1 << 31);
}

// D == 128, and 64 < D < 128 with the columns past D zero.
inline bool purified_d128_ok(const PurArgs& a) {
    return a.D > 64 && a.D <= 128 && a.doc == nullptr && ((int64_t)a.T + 256) * a.D * 2 < ((int64_t)1 << 31);
}

// 64 < D <= 128 with document ids: the D = 128 kernels' document mode (zero
// columns past D).
inline bool purified_d128_doc_ok(const PurArgs& a) {
    return a.D > 64 && a.D <= 128 && purified_window_ok(a) && a.doc != nullptr &&
           ((int64_t)a.T + 256) * a.D * 2 < ((int64_t)1 << 31);
}

inline bool purified_d256_ok(const PurArgs& a) {
    return a.D > 128 && a.D <= 256 && (a.doc == nullptr || purified_window_ok(a)) &&
           ((int64_t)a.T + 256) * a.D * 2 < ((int64_t)1 << 31);
}

inline bool purified_doc_fast_ok(const PurArgs& a) {
    return a.D == 64 && purified_window_ok(a) && a.doc != nullptr && ((int64_t)a.T + 256) * a.D * 2 < ((int64_t)1 << 31);
}

}  // namespace qdl
