// Purified-Born forward kernel instantiations: element type x padded head dim
// (32, 64, 128, 256; the host zero-pads D to a multiple of 8 and the kernels
// bound-check columns past D).
#include "born_fwd_d128.h"
#include "born_fwd_doc.h"
#include "born_launch.h"
#include "purified_dispatch.h"

namespace qdl {

template <class IN>
static hipError_t purified_fwd_dispatch(const PurArgs& a, hipStream_t s) {
    // 16-bit inputs, D <= 128: the 16-bit-MFMA kernels with each weight split
    // into two bf16 terms for P.V (fp16: the overlap on the fp16 MFMA, V split
    // exactly into two bf16 terms).
    using E = typename std::conditional<std::is_same<IN, F16>::value, F16, BF16>::type;
    constexpr bool k16 = !std::is_same<IN, float>::value;
    if constexpr (k16)
        if (purified_split_ok<IN>(a) && split16_pays(a, false, true)) return split16_fwd<E>(a, s);
    // D = 64 (and below, zero columns), dense, causal or a window.
    if (k16 && purified_fast_ok(a)) {
        if (a.window > 0)
            return a.is_causal ? launch_purified_fwd_fast<kWindow, false, E>(a, s)
                               : launch_purified_fwd_fast<kWindowNC, false, E>(a, s);
        return a.is_causal ? launch_purified_fwd_fast<kCausal, false, E>(a, s)
                           : launch_purified_fwd_fast<kDense, false, E>(a, s);
    }
    if (k16 && purified_narrow_ok(a)) {
        if (a.window > 0)
            return a.is_causal ? launch_purified_fwd_fast<kWindow, true, E>(a, s)
                               : launch_purified_fwd_fast<kWindowNC, true, E>(a, s);
        return a.is_causal ? launch_purified_fwd_fast<kCausal, true, E>(a, s)
                           : launch_purified_fwd_fast<kDense, true, E>(a, s);
    }
    // 64 < D <= 128, dense, causal or a window: the D = 128 kernel's purified
    // mode.
    if (k16 && purified_d128_ok(a)) {
        if (a.D == 128) {
            if (a.window > 0)
                return a.is_causal ? launch_purified_fwd_d128<kWindow, false, E>(a, s)
                                   : launch_purified_fwd_d128<kWindowNC, false, E>(a, s);
            return a.is_causal ? launch_purified_fwd_d128<kCausal, false, E>(a, s)
                               : launch_purified_fwd_d128<kDense, false, E>(a, s);
        }
        if (a.window > 0)
            return a.is_causal ? launch_purified_fwd_d128<kWindow, true, E>(a, s)
                               : launch_purified_fwd_d128<kWindowNC, true, E>(a, s);
        return a.is_causal ? launch_purified_fwd_d128<kCausal, true, E>(a, s)
                           : launch_purified_fwd_d128<kDense, true, E>(a, s);
    }
    // D = 128, document ids (with or without a causal window): its document
    // mode.
    if (k16 && purified_d128_doc_ok(a)) {
        if (a.D < 128) {
            if (a.window > 0) return launch_purified_fwd_d128_doc<kWindow, E, true>(a, s);
            return a.is_causal ? launch_purified_fwd_d128_doc<kCausal, E, true>(a, s)
                               : launch_purified_fwd_d128_doc<kDense, E, true>(a, s);
        }
        if (a.window > 0) return launch_purified_fwd_d128_doc<kWindow, E>(a, s);
        return a.is_causal ? launch_purified_fwd_d128_doc<kCausal, E>(a, s)
                           : launch_purified_fwd_d128_doc<kDense, E>(a, s);
    }
    // D = 64, document ids (with or without a causal window): the document
    // kernel's purified mode.
    if (k16 && purified_doc_fast_ok(a))
        return a.window > 0 ? launch_purified_fwd_doc<true, E>(a, s) : launch_purified_fwd_doc<false, E>(a, s);
    // Above D = 128, and documents at other head dims: the generic
    // 16-bit-MFMA kernels' purified mode.
    if (k16 && purified_d256_ok(a)) return purified_fwd_d256_launch(E::kDtype, a, s);
    if (k16 && (a.D > 128 || a.doc != nullptr)) return purified_wide_fwd_launch(E::kDtype, a, s);
    if (!k16 && purified_split_ok<IN>(a) &&
        !f32_staged(true, false, (int64_t)a.B * a.H, a.T, a.D, a.is_causal != 0, a.window,
                    a.doc != nullptr))
        return purified_fwd_f32_launch(a, s);
    switch (purified_padded_dim(a.D)) {
        case 32: return launch_purified_fwd<IN, 32>(a, s);
        case 64: return launch_purified_fwd<IN, 64>(a, s);
        case 128: return launch_purified_fwd<IN, 128>(a, s);
        default: return launch_purified_fwd<IN, 256>(a, s);
    }
}
// dtype codes as in qdl_flash_born.h: 0 fp32, 1 fp16, 2 bf16.
hipError_t purified_fwd_launch(int dtype, const PurArgs& a, hipStream_t s) {
    if (dtype == 0) return purified_fwd_dispatch<float>(a, s);
    if (dtype == 1) return purified_fwd_dispatch<F16>(a, s);
    return purified_fwd_dispatch<BF16>(a, s);
}

}  // namespace qdl
