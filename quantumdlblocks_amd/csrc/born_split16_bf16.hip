// Few-block kernel instantiations for bf16 inputs (born_split16.h).
#include "born_split16.h"
#include "born_launch.h"

namespace qdl {

template <>
hipError_t split16_fwd<BF16>(const FwdArgs& a, hipStream_t s) { return launch_split16_fwd<BF16, false>(a, s); }
template <>
hipError_t split16_fwd<BF16>(const PurArgs& a, hipStream_t s) { return launch_split16_fwd<BF16, true>(a, s); }
template <>
hipError_t split16_bwd<BF16>(const BwdArgs& a, hipStream_t s) { return launch_split16_bwd<BF16, false>(a, s); }
template <>
hipError_t split16_bwd<BF16>(const PurArgs& a, hipStream_t s) { return launch_split16_bwd<BF16, true>(a, s); }

}  // namespace qdl
