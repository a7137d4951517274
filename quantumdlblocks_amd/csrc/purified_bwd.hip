// Purified-Born backward kernel instantiations: element type x padded head dim
// (32, 64, 128, 256; the host zero-pads D to a multiple of 8 and the kernels
// bound-check columns past D).
#include "born_bwd_d128.h"
#include "born_bwd_fast.h"
#include "born_launch.h"
#include "purified_dispatch.h"

namespace qdl {

// 16-bit, D = 64: the 16-bit-MFMA dQ kernel (which also writes -delta and
// 1/Z) before the dK/dV kernel (which writes the dgamma / dtau partials), then
// the fixed-order reduction.  E: the input dtype, to which the reference
// rounds p/Z and dR before their contractions (flash_born.py:926, 939, 1058).
template <int MODE, bool DOC = false, bool PAD = false, class E = BF16>
static hipError_t purified_bwd_fast(const PurArgs& a, hipStream_t s) {
    // dQ: 256-row blocks of 4 waves, 128-row blocks of 2 with documents.
    constexpr int NW = DOC ? 2 : 4;
    hipLaunchKernelGGL((born_bwd16_dq_fast_kernel<E, 64, MODE, true, DOC, PAD, NW>),
                       dim3((unsigned)bwd16_dq_fast_groups(a.B, a.H, a.T, DOC)), dim3(64 * NW), 0, s, a);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const int nwg = purified_dkdv_groups(a.B, a.H, a.T, 64);
    hipLaunchKernelGGL((born_bwd16_dkdv_fast_kernel<E, 64, MODE, true, DOC, PAD>), dim3((unsigned)nwg), dim3(256), 0,
                       s, a);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    return launch_purified_param_reduce(a, nwg, s);
}

// 16-bit, 64 < D <= 128: the D = 128 dQ and dK/dV kernels' purified mode,
// then the same reduction.
template <int MODE, bool DOC = false, class E = BF16>
static hipError_t purified_bwd_d128(const PurArgs& a, hipStream_t s) {
    hipError_t e = a.D == 128 ? launch_purified_bwd_d128<MODE, false, DOC, E>(a, s)
                              : launch_purified_bwd_d128<MODE, true, DOC, E>(a, s);
    if (e != hipSuccess) return e;
    // dK/dV workgroups: 128-key blocks, 64-key blocks with documents.
    const int nwg = DOC ? ((a.T + 63) / 64) * a.B * a.H : purified_dkdv_groups(a.B, a.H, a.T, 128);
    return launch_purified_param_reduce(a, nwg, s);
}

template <class IN>
static hipError_t purified_bwd_dispatch(const PurArgs& a, hipStream_t s) {
    // 16-bit inputs: the 16-bit-MFMA backward kernels (bf16 and fp16 alike:
    // the reference rounds p/Z and dR to the input dtype before its dots).
    using E = typename std::conditional<std::is_same<IN, F16>::value, F16, BF16>::type;
    constexpr bool k16 = !std::is_same<IN, float>::value;
    if constexpr (k16) {
        if (purified_split_ok<IN>(a) && split16_pays(a, true, true)) {
            const hipError_t e = split16_bwd<E>(a, s);
            return e != hipSuccess ? e : launch_purified_param_reduce(a, f32_groups(a.B, a.H, a.T), s);
        }
    }
    if (k16 && purified_fast_ok(a)) {
        if (a.window > 0)
            return a.is_causal ? purified_bwd_fast<kWindow, false, false, E>(a, s)
                               : purified_bwd_fast<kWindowNC, false, false, E>(a, s);
        return a.is_causal ? purified_bwd_fast<kCausal, false, false, E>(a, s)
                           : purified_bwd_fast<kDense, false, false, E>(a, s);
    }
    if (k16 && purified_narrow_ok(a)) {
        if (a.window > 0)
            return a.is_causal ? purified_bwd_fast<kWindow, false, true, E>(a, s)
                               : purified_bwd_fast<kWindowNC, false, true, E>(a, s);
        return a.is_causal ? purified_bwd_fast<kCausal, false, true, E>(a, s)
                           : purified_bwd_fast<kDense, false, true, E>(a, s);
    }
    if (k16 && purified_d128_ok(a)) {
        if (a.window > 0)
            return a.is_causal ? purified_bwd_d128<kWindow, false, E>(a, s) : purified_bwd_d128<kWindowNC, false, E>(a, s);
        return a.is_causal ? purified_bwd_d128<kCausal, false, E>(a, s) : purified_bwd_d128<kDense, false, E>(a, s);
    }
    if (k16 && purified_d128_doc_ok(a)) {
        if (a.window > 0) return purified_bwd_d128<kWindow, true, E>(a, s);
        return a.is_causal ? purified_bwd_d128<kCausal, true, E>(a, s) : purified_bwd_d128<kDense, true, E>(a, s);
    }
    // D = 64, document ids (with or without a causal window): the same
    // kernels' document variants.
    if (k16 && purified_doc_fast_ok(a)) {
        if (a.window > 0) return purified_bwd_fast<kWindow, true, false, E>(a, s);
        return a.is_causal ? purified_bwd_fast<kCausal, true, false, E>(a, s)
                           : purified_bwd_fast<kDense, true, false, E>(a, s);
    }
    if (k16 && purified_d256_ok(a)) {
        hipError_t e = purified_bwd_d256_launch(E::kDtype, a, s);
        if (e != hipSuccess) return e;
        const int nwg = ((a.T + 127) / 128) * a.B * a.H;
        return launch_purified_param_reduce(a, nwg, s);
    }
    if (k16 && (a.D > 128 || a.doc != nullptr)) return purified_wide_bwd_launch(E::kDtype, a, s);
    if (!k16 && purified_split_ok<IN>(a) &&
        !f32_staged(true, true, (int64_t)a.B * a.H, a.T, a.D, a.is_causal != 0, a.window,
                    a.doc != nullptr))
        return purified_bwd_f32_launch(a, s);
    switch (purified_padded_dim(a.D)) {
        case 32: return launch_purified_bwd<IN, 32>(a, s);
        case 64: return launch_purified_bwd<IN, 64>(a, s);
        case 128: return launch_purified_bwd<IN, 128>(a, s);
        default: return launch_purified_bwd<IN, 256>(a, s);
    }
}

// dtype codes as in qdl_flash_born.h: 0 fp32, 1 fp16, 2 bf16.
hipError_t purified_bwd_launch(int dtype, const PurArgs& a, hipStream_t s) {
    if (dtype == 0) return purified_bwd_dispatch<float>(a, s);
    if (dtype == 1) return purified_bwd_dispatch<F16>(a, s);
    return purified_bwd_dispatch<BF16>(a, s);
}
int64_t purified_bwd_workspace_bytes(int dtype, int64_t B, int64_t H, int64_t T, int64_t D) {
    const int64_t region = (B * H * T * 4 + 255) / 256 * 256;
    // 32-key blocks (fp32 and few-block launches; never fewer than the others').
    (void)dtype;
    (void)D;
    const int64_t nwg = (T + 31) / 32 * B * H;
    return 2 * region + (2 * nwg * 4 + 255) / 256 * 256;
}

}  // namespace qdl
