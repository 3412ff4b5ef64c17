// The Dense projection kernels for bf16 payloads.
#include "gemm_dense.hpp"

namespace xp {

template struct DenseKernels<Bf16Payload>;

}  // namespace xp
