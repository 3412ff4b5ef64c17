// The grouped MoE projection kernels for bf16 payloads.
#include "gemm_grouped.hpp"

namespace xp {

template struct GroupedKernels<Bf16Payload>;

}  // namespace xp
