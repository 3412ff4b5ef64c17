// The biased projection kernels for bf16 payloads.
#include "gemm_extended.hpp"

namespace xp {

template struct ExtendedKernels<Bf16Payload>;

}  // namespace xp
