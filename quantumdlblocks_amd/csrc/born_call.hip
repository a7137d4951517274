// C ABI, struct form: qdl_flash_born_forward_call / _backward_call (declared
// in include/qdl_flash_born.h).  One argument block for the Born and purified
// kernels and the fused prologue; scale and tau by value or in device memory,
// gradients of the parameters only where asked for.
#include <stdint.h>

#include "../../include/qdl_flash_born.h"
#include "born_launch.h"
#include "purified_args.h"

namespace qdl {
hipError_t purified_fwd_launch(int dtype, const PurArgs& a, hipStream_t s);
hipError_t purified_bwd_launch(int dtype, const PurArgs& a, hipStream_t s);
int64_t purified_bwd_workspace_bytes(int dtype, int64_t B, int64_t H, int64_t T, int64_t D);
}  // namespace qdl

namespace {

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int hip_status(hipError_t e) { return e == hipSuccess ? QDL_BORN_OK : (int)e; }

// The checks of the positional entry points, on the block's fields.
int check(const qdl_born_call* c) {
    if (!c) return QDL_BORN_E_NULL;
    if (c->struct_bytes != (int64_t)sizeof(qdl_born_call)) return QDL_BORN_E_SHAPE;
    if (c->dtype != QDL_BORN_DTYPE_F32 && c->dtype != QDL_BORN_DTYPE_F16 && c->dtype != QDL_BORN_DTYPE_BF16)
        return QDL_BORN_E_DTYPE;
    if (c->B < 0 || c->H < 0 || c->T < 0) return QDL_BORN_E_SHAPE;
    if (c->B * c->H > (int64_t)1 << 24 || c->T > (int64_t)1 << 28 || c->B * c->H * c->T > ((int64_t)1 << 31) - 1)
        return QDL_BORN_E_SHAPE;
    if (c->D < 8 || c->D > 256 || c->D % 8 != 0) return QDL_BORN_E_HEADDIM;
    if (c->scale && c->n_scale != 1 && c->n_scale != c->H) return QDL_BORN_E_SCALE;
    if (c->purified && c->tau && c->n_tau != 1 && c->n_tau != c->H) return QDL_BORN_E_TAU;
    if (c->window_size < 0 || c->window_size > ((int64_t)1 << 30)) return QDL_BORN_E_WINDOW;
    if (!(c->eps >= 0.0)) return QDL_BORN_E_SHAPE;
    if (c->purified && !(c->eps_base == c->eps_base)) return QDL_BORN_E_SHAPE;
    return QDL_BORN_OK;
}

// The fields that FwdArgs, BwdArgs and PurArgs share.
template <class A>
void fill(A& a, const qdl_born_call* c) {
    a.q = c->q;
    a.k = c->k;
    a.v = c->v;
    a.scale = c->scale;
    a.scale_value = (float)c->scale_value;
    a.per_head_scale = c->scale && c->n_scale > 1 ? 1 : 0;
    a.doc = c->doc_ids;
    a.B = (int)c->B;
    a.H = (int)c->H;
    a.T = (int)c->T;
    a.D = (int)c->D;
    a.is_causal = c->is_causal ? 1 : 0;
    a.window = (int)c->window_size;
    a.eps = (float)c->eps;
}

void fill_purified(qdl::PurArgs& a, const qdl_born_call* c) {
    fill(a, c);
    a.tau = c->tau;
    a.tau_value = (float)c->tau_value;
    a.per_head_tau = c->tau && c->n_tau > 1 ? 1 : 0;
    a.eps_base = (float)c->eps_base;
}

}  // namespace

extern "C" {

int qdl_flash_born_forward_call(const qdl_born_call* c, qdl_stream_t stream) {
    int rc = check(c);
    if (rc != QDL_BORN_OK) return rc;
    if (c->B * c->H * c->T == 0) return QDL_BORN_OK;
    // The purified output in the element type: 16-bit inputs.
    const bool has16 = c->purified && c->out16;
    if (has16 && c->dtype == QDL_BORN_DTYPE_F32) return QDL_BORN_E_DTYPE;
    if (!c->q || !c->k || !c->v || (!c->out && !has16) || !c->z) return QDL_BORN_E_NULL;
    if (has16 && !aligned16(c->out16)) return QDL_BORN_E_ALIGN;
    if (c->prologue) {
        if (c->cos_table && (!c->sin_table || c->n_freq < 0 || c->n_freq > c->D / 2 || c->table_ld < c->n_freq))
            return QDL_BORN_E_TABLE;
        if (c->purified || !(c->norm_eps >= 0.0)) return QDL_BORN_E_SHAPE;
        if (!c->q_out || !c->k_out) return QDL_BORN_E_NULL;
        if (!aligned16(c->q_out) || !aligned16(c->k_out)) return QDL_BORN_E_ALIGN;
    } else if (!aligned16(c->q) || !aligned16(c->k)) {
        return QDL_BORN_E_ALIGN;
    }
    if (!aligned16(c->v) || !aligned16(c->out)) return QDL_BORN_E_ALIGN;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (c->purified) {
        qdl::PurArgs a = {};
        fill_purified(a, c);
        a.o = static_cast<float*>(c->out);
        a.o16 = c->out16;
        a.z = c->z;
        a.param_grads = c->param_grads ? 1 : 0;
        return hip_status(qdl::purified_fwd_launch((int)c->dtype, a, s));
    }
    qdl::FwdArgs a = {};
    fill(a, c);
    a.o = c->out;
    a.z = c->z;
    if (c->prologue) {
        const qdl::ProloguePlan p = {c->q_strides, c->k_strides, c->cos_table, c->sin_table, c->n_freq, c->table_ld,
                                     c->norm_eps,  c->q_out,     c->k_out,     c->q_rinv,    c->k_rinv};
        return qdl::fwd_with_prologue((int)c->dtype, a, p, s);
    }
    switch (c->dtype) {
        case QDL_BORN_DTYPE_BF16: return hip_status(qdl::fwd_launch_bf16(a, s));
        case QDL_BORN_DTYPE_F16: return hip_status(qdl::fwd_launch_f16(a, s));
        default: return hip_status(qdl::fwd_launch_f32(a, s));
    }
}

int qdl_flash_born_backward_call(const qdl_born_call* c, qdl_stream_t stream) {
    int rc = check(c);
    if (rc != QDL_BORN_OK) return rc;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (c->B * c->H * c->T == 0) {
        // Empty problem: the only outputs with elements are the parameters'.
        hipError_t e = hipSuccess;
        if (c->dscale) e = qdl::zero_fill(c->dscale, c->scale ? c->n_scale : 1, s);
        if (e == hipSuccess && c->dtau) e = qdl::zero_fill(c->dtau, c->tau ? c->n_tau : 1, s);
        return hip_status(e);
    }
    if (!c->q || !c->k || !c->v || !c->out || !c->dout || !c->z || !c->dq || !c->dk || !c->dv) return QDL_BORN_E_NULL;
    if (!aligned16(c->q) || !aligned16(c->k) || !aligned16(c->v) || !aligned16(c->out) || !aligned16(c->dout) ||
        !aligned16(c->dq) || !aligned16(c->dk) || !aligned16(c->dv))
        return QDL_BORN_E_ALIGN;
    const int64_t need = c->purified ? qdl::purified_bwd_workspace_bytes((int)c->dtype, c->B, c->H, c->T, c->D)
                                     : qdl::bwd_workspace_bytes(c->B, c->H, c->T);
    if (!c->workspace || c->workspace_bytes < need) return QDL_BORN_E_WORKSPACE;
    if (!aligned16(c->workspace)) return QDL_BORN_E_ALIGN;
    if (c->purified) {
        qdl::PurArgs a = {};
        fill_purified(a, c);
        a.o_in = static_cast<const float*>(c->out);
        a.dout = c->dout;
        a.z_in = c->z;
        a.dq = c->dq;
        a.dk = c->dk;
        a.dv = c->dv;
        a.dscale = c->dscale;
        a.dtau = c->dtau;
        a.param_grads = c->dscale || c->dtau ? 1 : 0;
        const int64_t region = qdl::bwd_region_bytes(c->B, c->H, c->T);
        char* w = static_cast<char*>(c->workspace);
        a.ndelta = reinterpret_cast<float*>(w);
        a.zinv = reinterpret_cast<float*>(w + region);
        a.part = reinterpret_cast<float*>(w + 2 * region);
        return hip_status(qdl::purified_bwd_launch((int)c->dtype, a, s));
    }
    qdl::BwdArgs a = {};
    fill(a, c);
    a.o = c->out;
    a.dout = c->dout;
    a.z = c->z;
    a.dq = c->dq;
    a.dk = c->dk;
    a.dv = c->dv;
    a.dscale = c->dscale;
    qdl::bwd_workspace_carve(c->workspace, c->B, c->H, c->T, &a.ndelta, &a.delta_z, &a.zinv, &a.dscale_part);
    switch (c->dtype) {
        case QDL_BORN_DTYPE_BF16: return hip_status(qdl::bwd_launch_bf16(a, s));
        case QDL_BORN_DTYPE_F16: return hip_status(qdl::bwd_launch_f16(a, s));
        default: return hip_status(qdl::bwd_launch_f32(a, s));
    }
}

}  // extern "C"
