// Definitions of the Dense kernel tables, for the translation units that instantiate them.
#pragma once

#include "gemm_tables.hpp"

namespace xp {

template <class Kernel>
const void *kernel_address(Kernel kernel) {
  return reinterpret_cast<const void *>(kernel);
}

template <class P>
const void *DenseKernels<P>::split(bool gated, int groups, bool gather) {
  if (gather) {
    return gated ? kernel_address(&split_gemm_kernel<split_depth(1), 1, true, true, P>)
                 : kernel_address(&split_gemm_kernel<split_depth(1), 1, false, true, P>);
  }
  if (groups == 1) {
    return gated ? kernel_address(&split_gemm_kernel<split_depth(1), 1, true, false, P>)
                 : kernel_address(&split_gemm_kernel<split_depth(1), 1, false, false, P>);
  }
  return gated ? kernel_address(&split_gemm_kernel<split_depth(2), 2, true, false, P>)
               : kernel_address(&split_gemm_kernel<split_depth(2), 2, false, false, P>);
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

template <bool GATED, class P>
const void *tile_kernel(int variant, bool stream) {
  using Kernel = void (*)(GemmArgs);
  static const Kernel table[][2] = {
      {&tile_gemm_kernel<256, 256, 2, 4, 2, GATED, false, false, P>, &tile_gemm_kernel<256, 256, 2, 4, 2, GATED, false, true, P>},
      {&tile_gemm_kernel<256, 128, 4, 2, 3, GATED, false, false, P>, &tile_gemm_kernel<256, 128, 4, 2, 3, GATED, false, true, P>},
      {&tile_gemm_kernel<128, 128, 2, 2, 3, GATED, false, false, P>, &tile_gemm_kernel<128, 128, 2, 2, 3, GATED, false, true, P>},
      {&tile_gemm_kernel<64, 128, 2, 2, 6, GATED, false, false, P>, &tile_gemm_kernel<64, 128, 2, 2, 6, GATED, false, true, P>},
      {&tile_gemm_kernel<64, 64, 2, 1, 4, GATED, false, false, P>, &tile_gemm_kernel<64, 64, 2, 1, 4, GATED, false, true, P>},
  };
  static_assert(sizeof(table) / sizeof(table[0]) == kTileShapeCount, "one kernel per tile shape");
  return kernel_address(table[variant][stream ? 1 : 0]);
}

template <class P>
const void *DenseKernels<P>::tile(bool gated, int variant, bool stream) {
  return gated ? tile_kernel<true, P>(variant, stream) : tile_kernel<false, P>(variant, stream);
}

}  // namespace xp
