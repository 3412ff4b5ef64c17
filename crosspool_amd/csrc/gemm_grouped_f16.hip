// The grouped MoE projection kernels for fp16 payloads.
#include "gemm_grouped.hpp"

namespace xp {

template struct GroupedKernels<F16Payload>;

}  // namespace xp
