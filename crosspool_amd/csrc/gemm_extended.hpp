// Definitions of the biased projections' kernel tables, for the translation units that
// instantiate them.
#pragma once

#include "gemm_tables.hpp"

namespace xp {

template <bool GATED, class P>
const void *extended_tile_kernel(int variant) {
  using Kernel = void (*)(GemmArgs);
  static const Kernel table[] = {
      &tile_gemm_kernel<256, 256, 2, 4, 2, GATED, false, false, P, true>,
      &tile_gemm_kernel<256, 128, 4, 2, 3, GATED, false, false, P, true>,
      &tile_gemm_kernel<128, 128, 2, 2, 3, GATED, false, false, P, true>,
      &tile_gemm_kernel<64, 128, 2, 2, 6, GATED, false, false, P, true>,
  };
  static_assert(sizeof(table) / sizeof(table[0]) == kExtendedTileShapes, "one kernel per shape");
  return reinterpret_cast<const void *>(table[variant]);
}

template <class P>
const void *ExtendedKernels<P>::tile(bool gated, int variant) {
  return gated ? extended_tile_kernel<true, P>(variant) : extended_tile_kernel<false, P>(variant);
}

}  // namespace xp
