// Backward kernel instantiations for fp32 inputs (Born; purified up to D = 128).
#include "born_bwd.h"
#include "born_f32.h"
#include "born_launch.h"
#include "purified_dispatch.h"

namespace qdl {

hipError_t bwd_launch_f32(const BwdArgs& a, hipStream_t s) {
    if (!f32_staged(false, true, (int64_t)a.B * a.H, a.T, a.D, a.is_causal != 0, a.window,
                    a.doc != nullptr)) {
        const hipError_t e = launch_f32_bwd<false>(a, s);
        return e != hipSuccess ? e : launch_bwd_common_post(a, s);
    }
    const int dp = padded_head_dim(a.D);
    const int mode = mask_mode(a.is_causal, a.window, a.doc);
    if (dp == 128) return mode == kDense ? launch_bwd32<128, kDense>(a, s) : launch_bwd32<128, kGeneral>(a, s);
#define QDL_MODE_BODY(M) return launch_bwd32<DPV, M>(a, s);
#define QDL_DP_BODY(D_) { constexpr int DPV = D_; QDL_SWITCH_MODE(mode, QDL_MODE_BODY) }
    QDL_SWITCH_DP_WIDE(dp, QDL_DP_BODY)
#undef QDL_DP_BODY
#undef QDL_MODE_BODY
    return hipErrorInvalidValue;
}

hipError_t purified_bwd_f32_launch(const PurArgs& a, hipStream_t s) { return launch_f32_bwd<true>(a, s); }

}  // namespace qdl
