// The Dense projection kernels for fp16 payloads.
#include "gemm_dense.hpp"

namespace xp {

template struct DenseKernels<F16Payload>;

}  // namespace xp
