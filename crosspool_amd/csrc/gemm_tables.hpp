// Kernel tables of the projections: which instantiation serves a choice.  Every Dense and
// grouped MoE kernel is instantiated for both payload dtypes (bf16, fp16); each payload's
// Dense and grouped instantiations are a translation unit of their own (gemm_dense_*.hip,
// gemm_grouped_*.hip), so that they compile in parallel.
#pragma once

#include "gemm_kernels.hpp"

namespace xp {

// Chunks of loads in flight per wave of the split kernel, by token groups (the register
// budget of two workgroups per CU).
constexpr int split_depth(int groups) { return groups == 1 ? 4 : 3; }

// The resident kernel for 16 token rows (two groups of 8) and `cpw` chunks per wave (1 to
// 4), and for 32 (four groups, two chunks in flight per wave) as the gate_up of a Dense
// step with the gather fused.  Measured on MI355X, Qwen3 layers at 17-32 rows against the
// separate gather and the 64 x 64 tiles: 4B (19456 weight rows) 50.3 / 51.2 / 53.4 ->
// 45.6 / 46.7 / 49.4 us at 20 / 24 / 32 rows, 8B (24576) 71.9 / 72.4 / 74.0 -> 69.4 /
// 70.4 / 72.4; 1.7B (12288) and 0.6B (6144) within +-1 us either way, so four groups serve
// only projections of at least kResidentWideMinN weight rows.  (At 9-16 rows four groups
// were 1.2-4.3 us slower than two.)
constexpr int kResidentMaxChunksPerWave = 4;
constexpr int kResidentGroups = 2;
constexpr int kResidentWideGroups = 4;

struct TileShape {
  int bm;
  int bn;
  int waves;
  int stages;           // LDS slabs (STAGES - 1 of them in flight); one workgroup per CU
  double flops_per_us;  // one CU's rate on this shape with every CU busy, measured on MI355X
};
constexpr TileShape kTileShapes[] = {
    {256, 256, 8, 2, 4.6e6},
    {256, 128, 8, 3, 4.0e6},
    {128, 128, 4, 3, 3.4e6},
    {64, 128, 4, 6, 2.4e6},
    {64, 64, 2, 4, 1.2e6},
    {192, 256, 8, 2, 4.5e6},
    {128, 256, 8, 3, 4.2e6},
};
constexpr int kTileShapeCount = sizeof(kTileShapes) / sizeof(kTileShapes[0]);
// The cost model ranks the first four shapes.  The 64 x 64 gated tile (two waves, four
// stages, two workgroups per CU) replaces the 64 x 128 one for a one-token-tile grid that
// leaves CUs idle: twice the workgroups stream the weights.  Measured on MI355X with weights
// streamed cold: Qwen3-0.6B gate_up at 32 / 64 / 128 rows 11.2 / 12.0 / 11.8 -> 9.3 / 9.8 /
// 9.8 us (48-96 -> 96-192 workgroups), Qwen3-8B gate_up at 32 rows 44.5 -> 43.0 us.
constexpr int kRankedTileShapes = 4;
constexpr int kDecodeTile = 3;        // 64 x 128
constexpr int kNarrowDecodeTile = 4;  // 64 x 64

// Chunks in flight per wave of the grouped split kernel.  Its workgroups are short (a wave
// streams one 16-row block of one expert: 24 KB of Qwen3-30B-A3B's down projection), so
// the fixed cost of each (the tile table, the route slots, the first round trip) weighs
// more than the depth of its ring: at depth 2 the kernel takes at most 128 VGPRs and a SIMD
// holds four of its waves (depth 4, with half as many: 6 % slower at 8 and 32 tokens).
constexpr int kGroupedSplitDepth = 2;

// How a tile launch loads its weights, each its own instantiation (a per-load branch on an
// argument cost the loading waves ~2 % at 2048 rows).  Stream: the grid has one token tile, so
// each weight tile has one reader and its loads carry the nontemporal hint.  StreamRotated: the
// same from another slab of K in each workgroup, for weight rows a multiple of 8 KB apart (the
// kernel's ROTATE).
enum class WeightLoads : int { Shared = 0, Stream = 1, StreamRotated = 2 };
constexpr int kRotatedTileRows = 128;
constexpr int64_t kRotatedPitch = 4096;  // columns
// K ranges start a K split's workgroups at different slabs already: up to four ranges gain from
// the rotation, eight are even and sixteen lose.  Layers at 17 / 32 / 45 / 64 / 90 / 128 rows: hidden
// 8192, intermediate 4096 (gate_up in 4 ranges, down in 4 or 2) 58.8 / 60.1 / 61.2 / 63.0 / 68.9 /
// 77.4 -> 55.3 / 56.6 / 57.5 / 59.3 / 62.0 / 71.8 us; Qwen3-8B (down in 8) 67.8 / 71.9 / 67.6 /
// 70.6 / 78.8 / 85.4 against 68.0 / 72.0 / 67.7 / 70.7 / 78.5 / 84.4 with it; 1024 / 4096 (down in 16)
// 22.6 / 23.8 / 24.6 / 25.3 against 22.8 / 24.1 / 24.9 / 25.5 up to 64 rows.
constexpr int64_t kRotatedRanges = 4;

template <class P>
struct DenseKernels {
  // The split kernel for `groups` token groups of 8 (1 or 2); the fused gather takes one.
  // (Four groups, 32 tokens, were measured and dropped: the token pieces read from L2 for each
  // weight line then cost more than the tile kernels, 60-77 us against 41-43 us for Qwen3-8B
  // gate_up at 17-32 rows.)
  // `half`: on 8-row weight blocks.
  static const void *split(bool gated, int groups, bool gather, bool half);
  // The persistent split kernel with the gather fused (one token group).
  static const void *split_gathered(bool gated);
  static const void *stream(bool gated, bool gather);
  static const void *stream_reduce(bool gated);
  // Null for a combination without an instantiation (four groups serve gate_up with the
  // gather fused only).
  static const void *resident(bool gated, bool gather, int cpw, int groups);
  static const void *tile(bool gated, int variant, WeightLoads loads);
};

template <class P>
struct GroupedKernels {
  // `extended`: the EXTENDED epilogue (a bias or a ReLU / GELU activation), a separate
  // instantiation so that the SiLU projections without bias keep their code (the general
  // epilogue cost the 128-row gate_up tiles 3 % at 2048 tokens).
  static const void *tile(bool gated, MoeTile tile, bool extended);
  static const void *split(bool gated);
};

// The tile shapes of kTileShapes 0 to 3 with the EXTENDED epilogue, without a K split: a biased
// projection (`bias_stride` 0), gated ones with any activation.
constexpr int kExtendedTileShapes = 4;
template <class P>
struct ExtendedKernels {
  static const void *tile(bool gated, int variant);
};

extern template struct DenseKernels<Bf16Payload>;
extern template struct DenseKernels<F16Payload>;
extern template struct GroupedKernels<Bf16Payload>;
extern template struct GroupedKernels<F16Payload>;
extern template struct ExtendedKernels<Bf16Payload>;
extern template struct ExtendedKernels<F16Payload>;

}  // namespace xp
