// Definitions of the Dense kernel tables, for the translation units that instantiate them.
#pragma once

#include "gemm_tables.hpp"

namespace xp {

template <class Kernel>
const void *kernel_address(Kernel kernel) {
  return reinterpret_cast<const void *>(kernel);
}

template <class P, int HALVES>
const void *split_kernel(bool gated, int groups, bool gather) {
  if (gather) {
    return gated ? kernel_address(&split_gemm_kernel<split_depth(1), 1, true, true, P, HALVES>)
                 : kernel_address(&split_gemm_kernel<split_depth(1), 1, false, true, P, HALVES>);
  }
  if (groups == 1) {
    return gated ? kernel_address(&split_gemm_kernel<split_depth(1), 1, true, false, P, HALVES>)
                 : kernel_address(&split_gemm_kernel<split_depth(1), 1, false, false, P, HALVES>);
  }
  return gated ? kernel_address(&split_gemm_kernel<split_depth(2), 2, true, false, P, HALVES>)
               : kernel_address(&split_gemm_kernel<split_depth(2), 2, false, false, P, HALVES>);
}

template <class P>
const void *DenseKernels<P>::split(bool gated, int groups, bool gather, bool half) {
  return half ? split_kernel<P, 1>(gated, groups, gather) : split_kernel<P, 2>(gated, groups, gather);
}

template <class P>
const void *DenseKernels<P>::split_gathered(bool gated) {
  return gated ? kernel_address(&split_gathered_kernel<split_depth(1), true, P>)
               : kernel_address(&split_gathered_kernel<split_depth(1), false, P>);
}

template <class P>
const void *DenseKernels<P>::stream(bool gated, bool gather) {
  if (gather) {
    return gated ? kernel_address(&stream_gemm_kernel<true, true, P>) : nullptr;
  }
  return gated ? kernel_address(&stream_gemm_kernel<true, false, P>) : kernel_address(&stream_gemm_kernel<false, false, P>);
}

template <class P>
const void *DenseKernels<P>::stream_reduce(bool gated) {
  return gated ? kernel_address(&stream_reduce_kernel<true, P>) : kernel_address(&stream_reduce_kernel<false, P>);
}

template <int TG, bool GATED, bool GATHER, class P>
const void *resident_kernel(int cpw) {
  using Kernel = void (*)(GemmArgs);
  static const Kernel table[kResidentMaxChunksPerWave] = {
      &resident_gemm_kernel<TG, 1, GATED, GATHER, P>, &resident_gemm_kernel<TG, 2, GATED, GATHER, P>,
      &resident_gemm_kernel<TG, 3, GATED, GATHER, P>, &resident_gemm_kernel<TG, 4, GATED, GATHER, P>};
  return kernel_address(table[cpw - 1]);
}

template <class P>
const void *DenseKernels<P>::resident(bool gated, bool gather, int cpw, int groups) {
  if (groups == kResidentWideGroups) {
    return gated && gather ? resident_kernel<kResidentWideGroups, true, true, P>(cpw) : nullptr;
  }
  if (groups != kResidentGroups) {
    return nullptr;
  }
  if (gated) {
    return gather ? resident_kernel<kResidentGroups, true, true, P>(cpw)
                  : resident_kernel<kResidentGroups, true, false, P>(cpw);
  }
  return resident_kernel<kResidentGroups, false, false, P>(cpw);
}

template <int BM, int BN, int WAVES_M, int WAVES_N, int STAGES, bool GATED, class P>
const void *tile_kernel(WeightLoads loads) {
  if (loads == WeightLoads::Shared) {
    return kernel_address(&tile_gemm_kernel<BM, BN, WAVES_M, WAVES_N, STAGES, GATED, false, false, P>);
  }
  if constexpr (BM <= kRotatedTileRows) {
    if (loads == WeightLoads::StreamRotated) {
      return kernel_address(&tile_gemm_kernel<BM, BN, WAVES_M, WAVES_N, STAGES, GATED, false, true, P, false, true>);
    }
  }
  return kernel_address(&tile_gemm_kernel<BM, BN, WAVES_M, WAVES_N, STAGES, GATED, false, true, P>);
}

template <bool GATED, class P>
const void *tile_kernel(int variant, WeightLoads loads) {
  static_assert(kTileShapeCount == 7, "one kernel per tile shape");
  switch (variant) {
    case 0:
      return tile_kernel<256, 256, 2, 4, 2, GATED, P>(loads);
    case 1:
      return tile_kernel<256, 128, 4, 2, 3, GATED, P>(loads);
    case 2:
      return tile_kernel<128, 128, 2, 2, 3, GATED, P>(loads);
    case 3:
      return tile_kernel<64, 128, 2, 2, 6, GATED, P>(loads);
    case 4:
      return tile_kernel<64, 64, 2, 1, 4, GATED, P>(loads);
    case 5:
      return tile_kernel<192, 256, 2, 4, 2, GATED, P>(loads);
    case 6:
      return tile_kernel<128, 256, 2, 4, 3, GATED, P>(loads);
    default:
      return nullptr;
  }
}

template <class P>
const void *DenseKernels<P>::tile(bool gated, int variant, WeightLoads loads) {
  return gated ? tile_kernel<true, P>(variant, loads) : tile_kernel<false, P>(variant, loads);
}

}  // namespace xp
