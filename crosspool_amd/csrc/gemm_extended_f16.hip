// The biased projection kernels for fp16 payloads.
#include "gemm_extended.hpp"

namespace xp {

template struct ExtendedKernels<F16Payload>;

}  // namespace xp
