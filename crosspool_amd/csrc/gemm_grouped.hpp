// Definitions of the grouped MoE kernel tables, for the translation units that instantiate them.
#pragma once

#include "gemm_tables.hpp"

namespace xp {

template <bool GATED, class P, bool X>
const void *grouped_tile_kernel(MoeTile tile) {
  switch (tile) {
    case MoeTile::Rows64:
      return reinterpret_cast<const void *>(&tile_gemm_kernel<64, 128, 2, 2, 3, GATED, true, true, P, X>);
    case MoeTile::Rows128Stream:
      return GATED ? reinterpret_cast<const void *>(&tile_gemm_kernel<128, 256, 2, 4, 3, GATED, true, true, P, X>)
                   : reinterpret_cast<const void *>(&tile_gemm_kernel<128, 128, 4, 2, 2, GATED, true, true, P, X>);
    case MoeTile::Rows128:
      return GATED ? reinterpret_cast<const void *>(&tile_gemm_kernel<128, 256, 2, 4, 3, GATED, true, false, P, X>)
                   : reinterpret_cast<const void *>(&tile_gemm_kernel<128, 128, 4, 2, 2, GATED, true, false, P, X>);
    case MoeTile::Rows256:
      return reinterpret_cast<const void *>(&tile_gemm_kernel<256, 128, 4, 2, 3, GATED, true, true, P, X>);
    default:
      return nullptr;
  }
}

template <class P>
const void *GroupedKernels<P>::tile(bool gated, MoeTile tile, bool extended) {
  if (extended) {
    return gated ? grouped_tile_kernel<true, P, true>(tile) : grouped_tile_kernel<false, P, true>(tile);
  }
  return gated ? grouped_tile_kernel<true, P, false>(tile) : grouped_tile_kernel<false, P, false>(tile);
}

template <class P>
const void *GroupedKernels<P>::split(bool gated) {
  return gated ? reinterpret_cast<const void *>(&grouped_split_kernel<kGroupedSplitDepth, true, P>)
               : reinterpret_cast<const void *>(&grouped_split_kernel<kGroupedSplitDepth, false, P>);
}

}  // namespace xp
