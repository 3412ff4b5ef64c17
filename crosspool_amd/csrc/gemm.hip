// Kernel choice and launches of the projections: which kernel of gemm_kernels.hpp serves a
// row capacity and shape (choose_gemm, choose_dense_gate_up), and the launch records of that
// choice (make_gemm, make_grouped_gemm, make_grouped_split).

#include "gemm_tables.hpp"

#include <algorithm>
#include <mutex>

namespace xp {
namespace {

int split_groups(int64_t capacity) { return capacity <= kSplitGroupTokens ? 1 : 2; }

constexpr int kComputeUnits = 256;

// Decode sizes (up to 16 rows) take the split or the stream kernel, whichever a cost model
// in microseconds prefers.  Both stream the weights with 8-wave workgroups, each at a
// bounded rate (measured, the chip rate scales with the workgroup count up to the CU
// count), so a grid of few workgroups is the thing to avoid (Qwen3-4B down through the
// split kernel with 2 K ranges per row block has 80 workgroups: 41 us; with 8, 320: 16 us),
// workgroups past 256 run as further rounds, and the chip caps the total (both read whole
// 128-byte weight lines with the nontemporal hint).
// The split kernel reads its token pieces from L2, a little more per row and chunk of its
// K range; the stream kernel's K slices cost the reduction launch and their partial
// traffic.  The split kernel's rounds of 256 workgroups are priced one after another (each
// at the chip rate or at one workgroup's rate, whichever is slower, and never below one load
// round trip: short rounds are latency-bound).  Least-squares fit (relative error) to 498
// forced split (every K split) and stream (K slices of 512-4096 columns) timings on MI355X:
// the Qwen3 0.6B / 1.7B / 4B / 8B projections, the Qwen3-32B TP shard's and a hidden-1536
// down at 1 to 16 rows, the weights rotated over three copies (streamed from HBM).  Mean
// modelled error 7.4 % (26 % for the constants it replaced); summed over the 66
// (projection, rows) cases, its picks are 29 us slower than the fastest measured ones,
// against 79 us before.  Per layer (alternating builds on one box) that took the 9-16-row
// Dense steps of Qwen3-4B / 1.7B / the 32B shard from 47-51 / 34-38 / 42-47 us to 44-45 /
// 33-35 / 39-41 us and hidden 1536 at 1-8 rows from 27-31 to 26-27 us (Qwen3-8B at 9 rows:
// 61.4 -> 62.5 us, the one loss).
constexpr int64_t kDecodeMaxRows = 16;
constexpr int64_t kSplitMaxRows = kSplitGroupTokens * kSplitMaxGroups;
// Index: token groups - 1.  Two groups read twice the token pieces from L2 per weight line,
// which lowers the chip rate.
constexpr double kSplitWorkgroupBytesPerUs[kSplitMaxGroups] = {32.7e3, 27.6e3};
constexpr double kSplitBytesPerUs[kSplitMaxGroups] = {6.75e6, 5.06e6};
constexpr double kSplitFixedUs[kSplitMaxGroups] = {3.54, 4.19};
constexpr double kSplitRoundFloorUs = 2.7;  // no round of workgroups is shorter (one load round trip)
constexpr double kSplitTieMargin = 0.001;
// Per row past the first and 128-wide chunk of a range (padded to the load depth).
constexpr double kSplitRowUsPerChunk[kSplitMaxGroups] = {0.0406, 0.0314};
constexpr double kStreamWorkgroupBytesPerUs = 29.2e3;
constexpr double kStreamBytesPerUs = 6.1e6;
constexpr double kStreamFixedUs = 1.03;
constexpr double kStreamRowUs = 0.0071;  // per row past the first and 512 columns of the K slice
constexpr double kStreamReduceUs = 5.4;  // the reduction launch (it also ends the overlap of slices)
constexpr double kStreamPartialBytesPerUs = 6.0e6;
constexpr int kSplitDepth = 4;
constexpr double kGatherUs = 4.0;  // a separate gather launch at decode sizes (measured 3.8-4.0 us)
// The split kernel's fused gather runs in every workgroup, one per CU (its registers allow
// no second), beside only the first weight chunks: measured 2.3 us per round of 256
// workgroups for Qwen3-0.6B gate_up (one round), 3.3 and 4.4 us for Qwen3-8B (3 and 6).
constexpr double kSplitGatherRoundUs = 3.0;
// The same for the stream kernel's fused gather, per round of workgroups (measured: Qwen3-8B
// gate_up at 16 rows, 192 workgroups, 37.0 us plain and ~41 us with the gather fused).
constexpr double kStreamGatherUs = 3.5;
constexpr int64_t kSplitGatherMaxK = 4096;  // 8 staged rows of K + 16 bf16 (66 KB) beside the partial sums
static_assert(kSplitGatherMaxK * 2 <= kSplitGatheredScratchBytes, "the norm weights fit the partial sums' space");
static_assert(kSplitGatherMaxK / 8 <= 8 * 64, "a staged row is at most 8 chunks per lane");
// split_gathered_kernel: two workgroups per CU (128 VGPRs; at most 80 KB of LDS each, the
// 8 staged rows of 4096 + 16 bf16 and the space shared by the norm weights and the partial
// sums), for projections with at least that many units.  Its gather runs under the first
// weight chunks' round trip and its token pieces come from LDS (no per-row L2 reads); what
// the gather still adds is the normalisation pass over LDS and one barrier: measured on
// MI355X, the Qwen3-8B / 4B / 1.7B layer at one row 52.2 / 36.9 / 24.7 us against 55.0 /
// 37.7 / 26.6 us when the gather took its own round trip before the weight stream.
constexpr int64_t kSplitGatheredWorkgroups = 2 * kComputeUnits;
constexpr double kSplitPersistentGatherUs = 1.0;

double decode_stream_us(int64_t n, int64_t k, int64_t workgroups, double workgroup_bytes_per_us,
                        double chip_bytes_per_us, double fixed_us) {
  const int64_t rounds = (workgroups + kComputeUnits - 1) / kComputeUnits;
  const double bytes = 2.0 * static_cast<double>(n) * static_cast<double>(k);
  const double per_workgroup = static_cast<double>(rounds) * bytes / workgroups / workgroup_bytes_per_us;
  const double chip = bytes / chip_bytes_per_us;
  return (per_workgroup > chip ? per_workgroup : chip) + fixed_us;
}

// Candidate K splits of the split kernel (1, 2, 4 or 8 ranges per 16-row block, each range
// a whole number of 128-wide chunks and none empty) and their modelled cost at `capacity`
// rows, with the gather fused when `gather` is set.
GemmChoice choose_split(int64_t capacity, int64_t n, int64_t k, double &cost, bool gather = false,
                        bool persistent = false) {
  const int64_t quantum = 128;
  const int64_t row_blocks = (n + 15) / 16;
  const int groups = split_groups(capacity);
  const int64_t depth = split_depth(groups);
  GemmChoice best{GemmKind::Split, groups, 0, 1};
  cost = -1.0;
  for (int64_t ksplit = 1; ksplit <= kSplitWaves; ksplit *= 2) {
    const int64_t slice = ((k + ksplit - 1) / ksplit + quantum - 1) / quantum * quantum;
    if ((ksplit - 1) * slice >= k) {
      break;
    }
    const int64_t workgroups = (row_blocks * ksplit + kSplitWaves - 1) / kSplitWaves;
    const double workgroup_bytes = 2.0 * static_cast<double>(n) * static_cast<double>(k) / workgroups;
    double us = kSplitFixedUs[groups - 1];
    for (int64_t left = workgroups; left > 0; left -= kComputeUnits) {
      const double round_bytes = static_cast<double>(left < kComputeUnits ? left : kComputeUnits) * workgroup_bytes;
      const double chip_us = round_bytes / kSplitBytesPerUs[groups - 1];
      const double workgroup_us = workgroup_bytes / kSplitWorkgroupBytesPerUs[groups - 1];
      const double round_us = chip_us > workgroup_us ? chip_us : workgroup_us;
      us += round_us > kSplitRoundFloorUs ? round_us : kSplitRoundFloorUs;
    }
    us += kSplitRowUsPerChunk[groups - 1] *
                    static_cast<double>((slice / 128 + depth - 1) / depth * depth) *
                    static_cast<double>(capacity - 1);
    if (gather) {
      us += kSplitGatherRoundUs * static_cast<double>((workgroups + kComputeUnits - 1) / kComputeUnits);
    }
    // The persistent kernel walks units on a fixed grid, so it takes the most K ranges of
    // at least two chunks (the most units to balance) rather than the cheapest round count.
    // Otherwise a split whose cost equals the cheapest so far (within kSplitTieMargin, i.e.
    // rounding) takes its place: the most ranges among equal costs, shorter per-wave load
    // chains (Qwen3-8B gate_up at one row: 4 and 8 ranges model the same, and 8 is the
    // persistent kernel's split).
    if (persistent ? slice >= 2 * quantum : (cost < 0.0 || us < cost * (1.0 + kSplitTieMargin))) {
      best = {GemmKind::Split, groups, slice, ksplit};
      cost = us;
    }
  }
  return best;
}

constexpr int64_t kStreamLdsBytes = 160 * 1024 - 256;  // the fused gather's row table is static LDS
constexpr int64_t kStreamSliceQuantum = 128 * kStreamDepth;  // a whole number of load groups

int64_t stream_slices(int64_t k, int64_t k_slice) { return (k + k_slice - 1) / k_slice; }

// K slice of the stream kernel: workgroups are (8 row blocks) x (one slice), and the slice
// count minimising the modelled cost wins.
GemmChoice choose_stream(int64_t capacity, int64_t n, int64_t k, double &cost) {
  constexpr int64_t tp = 16;  // staged token rows
  const int64_t groups = ((n + 15) / 16 + kStreamWaves - 1) / kStreamWaves;
  GemmChoice best{GemmKind::Stream, 0, 0, 1};
  cost = -1.0;
  for (int64_t slices = 1; slices <= 64; ++slices) {
    const int64_t k_slice = ((k + slices - 1) / slices + kStreamSliceQuantum - 1) / kStreamSliceQuantum *
                            kStreamSliceQuantum;
    if (tp * (k_slice + kStreamRowPad) * 2 > kStreamLdsBytes || stream_slices(k, k_slice) != slices) {
      continue;  // does not fit LDS, or the same slice length as fewer slices
    }
    double us = decode_stream_us(n, k, slices * groups, kStreamWorkgroupBytesPerUs, kStreamBytesPerUs, kStreamFixedUs) +
                kStreamRowUs * static_cast<double>(capacity - 1) * static_cast<double>(k_slice) / 512.0;
    if (slices > 1) {
      us += kStreamReduceUs + 8.0 * static_cast<double>(slices * capacity * n) / kStreamPartialBytesPerUs;
    }
    if (cost < 0.0 || us < cost) {
      best = {GemmKind::Stream, 0, k_slice, 1};
      cost = us;
    }
  }
  return best;
}

// Tile shape and K split for a projection at `capacity` rows, from a cost model in
// microseconds.  Compute: whole rounds of one tile per CU at the shape's measured rate.
// Weights: streamed from HBM once.  The two overlap only in part (the slower counts fully,
// the faster by half).  A K split adds its fp32 partial traffic and the reduction launch;
// it fills the CUs when the tile grid is smaller than the chip (the down projection has 16
// to 32 weight tiles at H = 4096).  Fitted to forced-choice timings of the Qwen3 0.6B /
// 4B / 8B / 32B-shard projections at 32 to 4096 rows (weights streamed from HBM at the
// HBM-bound sizes), where it picks the fastest measured choice or one within 7 % of it.
constexpr double kWeightBytesPerUs = 4.5e6;   // weights streamed from HBM by the tile kernel
constexpr double kPartialBytesPerUs = 6.0e6;  // partial sums written, then read by the reduction
constexpr double kReduceLaunchUs = 4.0;
constexpr double kOverlap = 0.5;              // share of the faster of compute and streaming exposed
constexpr int64_t kMaxTileSplit = 16;

// A column split: the first n1 weight rows on shape `main` in whole rounds of one tile per
// CU, the other n - n1 on shape `tail` in a second launch, where one shape alone ends in a
// partial round (Qwen3-32B TP shard at 8192 rows: gate_up 800 tiles of 256 x 256, 3.125
// rounds).  Taken when the model prices it at least kColumnSplitGain below the best single
// shape, which keeps the choice away from near ties.
constexpr double kTailLaunchUs = 3.0;
constexpr double kColumnSplitGain = 0.05;

double tile_rounds_us(const TileShape &shape, int64_t rounds, int64_t k) {
  return static_cast<double>(rounds) * 2.0 * shape.bm * shape.bn * static_cast<double>(k) / shape.flops_per_us;
}

GemmChoice choose_tile(int64_t capacity, int64_t n, int64_t k, bool split_columns) {
  GemmChoice best{GemmKind::Tile, 0, k, 1};
  double best_cost = 0.0;
  for (int index = 0; index < kRankedTileShapes; ++index) {
    const TileShape &shape = kTileShapes[index];
    const int64_t base_tiles = ((capacity + shape.bm - 1) / shape.bm) * ((n + shape.bn - 1) / shape.bn);
    for (int64_t split = 1; split <= kMaxTileSplit; split *= 2) {
      const int64_t k_slice = ((k + split - 1) / split + 63) / 64 * 64;
      if ((split - 1) * k_slice >= k) {
        break;  // the last range would be empty
      }
      const int64_t rounds = (base_tiles * split + kComputeUnits - 1) / kComputeUnits;
      const double compute = static_cast<double>(rounds) * 2.0 * shape.bm * shape.bn *
                             static_cast<double>(k_slice) / shape.flops_per_us;
      const double stream = 2.0 * static_cast<double>(n) * static_cast<double>(k) / kWeightBytesPerUs;
      double cost = compute > stream ? compute + kOverlap * stream : stream + kOverlap * compute;
      if (split > 1) {
        cost += 8.0 * split * static_cast<double>(capacity) * static_cast<double>(n) / kPartialBytesPerUs +
                kReduceLaunchUs;
      }
      if ((index == 0 && split == 1) || cost < best_cost) {
        best = {GemmKind::Tile, index, k_slice, split};
        best_cost = cost;
      }
    }
  }
  if (!split_columns) {
    return best;
  }
  const double stream = 2.0 * static_cast<double>(n) * static_cast<double>(k) / kWeightBytesPerUs;
  GemmChoice split_best = best;
  double split_cost = best_cost * (1.0 - kColumnSplitGain);
  // The first launch runs on the 256 x 256 tile, the most efficient shape: with a 256 x 128
  // first launch the split measured slower than the best single shape (Qwen3-8B gate_up at
  // 512 rows 177 -> 186 us, the 32B shard's down at 2048 rows 228 -> 234 us per layer).
  for (int main = 0; main < 1; ++main) {
    const TileShape &shape = kTileShapes[main];
    const int64_t token_tiles = (capacity + shape.bm - 1) / shape.bm;
    for (int64_t weight_tiles = 1; weight_tiles * shape.bn < n; ++weight_tiles) {
      if ((token_tiles * weight_tiles) % kComputeUnits != 0) {
        continue;  // the first launch must be whole rounds
      }
      const int64_t n1 = weight_tiles * shape.bn;
      for (int tail = 0; tail < kRankedTileShapes; ++tail) {
        const TileShape &other = kTileShapes[tail];
        const int64_t tail_tiles = ((capacity + other.bm - 1) / other.bm) * ((n - n1 + other.bn - 1) / other.bn);
        const double compute =
            tile_rounds_us(shape, token_tiles * weight_tiles / kComputeUnits, k) +
            tile_rounds_us(other, (tail_tiles + kComputeUnits - 1) / kComputeUnits, k) + kTailLaunchUs;
        const double cost = compute > stream ? compute + kOverlap * stream : stream + kOverlap * compute;
        if (cost < split_cost) {
          split_cost = cost;
          split_best = {GemmKind::Tile, main, k, 1};
          split_best.tail_variant = tail;
          split_best.tail_columns = n - n1;
        }
      }
    }
  }
  return split_best;
}

// The resident kernel's K parts and chunks per wave at `capacity` rows (9 to 16, or 17 to
// 32 for a projection with the gather fused and at least kResidentWideMinN weight rows, on
// four token groups), with its modelled cost in microseconds (-1: not applicable).  Every workgroup streams its blocks'
// columns of its part at one workgroup's rate after a fixed prologue (launch, the token
// pieces, the first weight round trip), and the busiest workgroup sets the time; more than
// one part adds the partial sums and the reduction launch.  With the gather fused the part
// must cover K (a row's sum of squares needs every column).  Least-squares fit (relative
// error) to the kernel's durations on MI355X for the Qwen3 0.6B / 1.7B / 4B / 8B gate_up
// (gather fused) and the Qwen3 1.7B / 4B / 8B and 32B TP-shard down projections at 9 and 16
// rows, weights streamed from HBM: within 10 %.  The weight rows must fill the grid (N of at
// least 2048: a Router projection's few experts do not).
constexpr int64_t kResidentMinRows = 9;
constexpr int64_t kResidentMaxRows = 8 * kResidentGroups;
constexpr int64_t kResidentWideMaxRows = 8 * kResidentWideGroups;
constexpr int64_t kResidentMinN = 2048;
constexpr int64_t kResidentWideMinN = 16384;
constexpr double kResidentWorkgroupBytesPerUs[2] = {35.7e3, 24.8e3};  // index: gather fused
constexpr double kResidentFixedUs[2] = {7.8, 8.0};

GemmChoice choose_resident(int64_t capacity, int64_t n, int64_t k, bool gather, double &cost) {
  const bool wide = gather && capacity > kResidentMaxRows && capacity <= kResidentWideMaxRows && n >= kResidentWideMinN;
  const int groups = wide ? kResidentWideGroups : kResidentGroups;
  GemmChoice best{GemmKind::Resident, groups, 0, 0};
  cost = -1.0;
  if (capacity < kResidentMinRows || (capacity > kResidentMaxRows && !wide) || n < kResidentMinN ||
      n * k * 2 > INT32_MAX) {
    return best;
  }
  const int64_t chunks = (k + kResidentChunk - 1) / kResidentChunk;
  const int64_t row_blocks = (n + 15) / 16;
  for (int cpw = 1; cpw <= kResidentMaxChunksPerWave; ++cpw) {
    const int64_t part_chunks = static_cast<int64_t>(kResidentWaves) * cpw;
    const int64_t parts = (chunks + part_chunks - 1) / part_chunks;
    if ((gather && parts > 1) || parts > kResidentWorkgroups) {
      continue;
    }
    const int64_t walkers = std::min<int64_t>(kResidentWorkgroups / parts, row_blocks);
    const int64_t blocks = (row_blocks + walkers - 1) / walkers;
    const double columns = static_cast<double>(std::min<int64_t>(part_chunks * kResidentChunk, k));
    double us = kResidentFixedUs[gather ? 1 : 0] +
                static_cast<double>(blocks) * 16.0 * columns * 2.0 / kResidentWorkgroupBytesPerUs[gather ? 1 : 0];
    if (parts > 1) {
      us += kStreamReduceUs + 8.0 * static_cast<double>(parts * capacity * n) / kStreamPartialBytesPerUs;
    }
    if (cost < 0.0 || us < cost * (1.0 - kSplitTieMargin)) {
      best = {GemmKind::Resident, groups, part_chunks * kResidentChunk, parts};
      cost = us;
    }
  }
  return best;
}

}  // namespace

// The split or the stream kernel for a decode size, whichever the cost model prefers, and
// its modelled cost in microseconds.
GemmChoice choose_decode(int64_t capacity, int64_t n, int64_t k, double &cost) {
  const GemmChoice split = choose_split(capacity, n, k, cost);
  if (capacity <= kDecodeMaxRows) {
    double stream_us = 0.0;
    const GemmChoice stream = choose_stream(capacity, n, k, stream_us);
    if (stream_us < cost) {
      cost = stream_us;
      return stream;
    }
  }
  return split;
}

GemmChoice choose_gemm(int64_t capacity, int64_t n, int64_t k, bool gated, bool split_columns) {
  // 9 to 16 rows: the resident kernel where its model is cheaper than the split / stream
  // choice's.  Measured on MI355X (kernel durations, weights streamed from HBM): the Qwen3-32B
  // TP shard's down at 9 / 16 rows 12.8 / 13.3 us + a 4.0 us reduction (stream, 8 slices)
  // -> 12.3 / 13.2 us (one part, no reduction); Qwen3-4B and 1.7B down stay on the stream
  // kernel (resident 14.2 / 10.7 us + reduction against 12.5 / 8.5 us + reduction).
  // The split, stream and resident kernels address the weights through one 32-bit buffer range.
  if (capacity <= kDecodeMaxRows && n * k * 2 <= INT32_MAX) {
    double decode_us = 0.0;
    const GemmChoice decode = choose_decode(capacity, n, k, decode_us);
    double resident_us = 0.0;
    const GemmChoice resident = choose_resident(capacity, n, k, false, resident_us);
    return resident_us >= 0.0 && resident_us < decode_us ? resident : decode;
  }
  GemmChoice choice = choose_tile(capacity, n, k, split_columns);
  // Token tiles more than half full carry twice the MFMA work per weight byte, which the
  // two-wave tile's lower matrix rate turns into a loss once its grid passes the CU count
  // (Qwen3-8B at 64 rows: 81.2 -> 82.7 us per layer; Qwen3-0.6B at 256 rows: 30.1 -> 31.7).
  const TileShape &decode = kTileShapes[kDecodeTile];
  const int64_t decode_tiles = ((capacity + decode.bm - 1) / decode.bm) * ((n + decode.bn - 1) / decode.bn);
  const int64_t weight = capacity > decode.bm / 2 ? 2 : 1;
  if (gated && choice.variant == kDecodeTile && choice.k_split == 1 && choice.tail_variant < 0 &&
      decode_tiles * weight < kComputeUnits) {
    choice.variant = kNarrowDecodeTile;
  }
  return choice;
}

// Tile, K split or column split of a Dense step's projection above kStepMinRows rows, from a
// model of one launch in microseconds: whole rounds of one tile per CU, each at the shape's
// full rate, and a last round whose slabs go the faster the fewer CUs it fills (the chip
// clocks higher and its L2s have fewer readers); the weights' stream adds to it, since a round's
// tiles wait for the same lines; a K split adds its reduction and its sums' traffic.  A
// column split is two such launches.
// Fitted (log least squares) to some 9500 forced choices on MI355X: Qwen3 0.6B / 1.7B / 4B / 8B, a
// hidden-1536 layer and the Qwen3-32B TP shard, both projections, 26 row counts from 65 to 4096,
// every shape and 1 to 16 K ranges, weights streamed from HBM: mean error 6.1 %, and its picks
// sum to 0.6 % above the fastest measured single launch of each.  The column splits it prices
// were measured too (183 of them); they cost 11 % more than two modelled launches plus
// kStepTailUs.  The choice for the template's capacity stays unless the model prices another
// kStepGain below it, about the model's error: over the same sweep that loses against it in one
// case (3.9 %) and sums to 1 % above the best, where choose_gemm's choices (which know neither
// 192 x 256 and 128 x 256 tiles nor K splits that are no power of two) sum to 6 % above.
struct StepTile {
  int variant;
  double slab_us;   // per 64 columns of a round, however full
  double fill_us;   // the same, times the share of the CUs the round fills
  double tile_us;   // prologue and epilogue of a round
};
constexpr StepTile kStepTiles[] = {
    {0, 1.091, 0.203, 4.50},  // 256 x 256
    {1, 0.544, 0.156, 3.21},  // 256 x 128
    {2, 0.412, 0.073, 2.97},  // 128 x 128
    {3, 0.272, 0.082, 2.35},  // 64 x 128
    {5, 0.999, 0.141, 3.62},  // 192 x 256
    {6, 0.612, 0.148, 3.24},  // 128 x 256
};
constexpr int64_t kStepMinRows = 65;
constexpr int64_t kStepSplits[] = {1, 2, 3, 4, 6, 8, 12, 16};
constexpr int64_t kStepMinSlabs = 3;  // per K range
constexpr double kStepLaunchUs = 2.42;
constexpr double kStepReduceUs = 4.21;
constexpr double kStepPartialBytesPerUs = 7.76e6;
constexpr double kStepWeightBytesPerUs = 16.7e6;
constexpr double kStepTailUs = 5.6;
constexpr double kStepTailScale = 1.11;
constexpr double kStepGain = 0.10;

// Compute time of one launch of `weight_tiles` x the token tiles x `splits` workgroups.
double step_compute_us(const StepTile &tile, int64_t capacity, int64_t n, int64_t slabs, int64_t splits) {
  const TileShape &shape = kTileShapes[tile.variant];
  const int64_t workgroups = (capacity + shape.bm - 1) / shape.bm * ((n + shape.bn - 1) / shape.bn) * splits;
  const int64_t rounds = workgroups / kComputeUnits;
  const double rest = static_cast<double>(workgroups - rounds * kComputeUnits) / kComputeUnits;
  const double columns = static_cast<double>(slabs);
  double us = static_cast<double>(rounds) * (columns * (tile.slab_us + tile.fill_us) + tile.tile_us);
  if (rest > 0.0) {
    us += columns * (tile.slab_us + tile.fill_us * rest) + tile.tile_us;
  }
  return us;
}

// The model's time of a tile choice at `rows` rows, or -1 where it has no figures (64 x 64).
double step_us(const GemmChoice &choice, int64_t rows, int64_t n, int64_t k, double tail_scale = kStepTailScale) {
  const StepTile *main = nullptr;
  const StepTile *tail = nullptr;
  for (const StepTile &tile : kStepTiles) {
    main = tile.variant == choice.variant ? &tile : main;
    tail = tile.variant == choice.tail_variant ? &tile : tail;
  }
  if (main == nullptr || (choice.tail_columns > 0 && tail == nullptr)) {
    return -1.0;
  }
  const int64_t slabs = (choice.k_slice + 63) / 64;
  double us = kStepLaunchUs + step_compute_us(*main, rows, n - choice.tail_columns, slabs, choice.k_split) +
              2.0 * static_cast<double>(n) * static_cast<double>(k) / kStepWeightBytesPerUs;
  if (choice.k_split > 1) {
    us += kStepReduceUs + 8.0 * static_cast<double>(choice.k_split * rows * n) / kStepPartialBytesPerUs;
  }
  if (choice.tail_columns > 0) {
    us = tail_scale * (us + step_compute_us(*tail, rows, choice.tail_columns, slabs, 1)) + kStepTailUs;
  }
  return us;
}

// The model's time of one launch over `splits` K ranges, or -1 where they would be too short or
// the last one empty.
double step_split_us(const StepTile &tile, int64_t rows, int64_t n, int64_t k, int64_t splits) {
  const int64_t slabs = (k + 63) / 64;
  const int64_t per_range = (slabs + splits - 1) / splits;
  if (splits > 1 && (per_range < kStepMinSlabs || (splits - 1) * per_range >= slabs)) {
    return -1.0;
  }
  const double stream = 2.0 * static_cast<double>(n) * static_cast<double>(k) / kStepWeightBytesPerUs;
  const double plane_us = 8.0 * static_cast<double>(rows * n) / kStepPartialBytesPerUs;
  return kStepLaunchUs + stream + step_compute_us(tile, rows, n, per_range, splits) +
         (splits > 1 ? kStepReduceUs + static_cast<double>(splits) * plane_us : 0.0);
}

// Whether choose_step_tile can take a K split: none of its unsplit launches is cheaper.
bool step_split_pays(int64_t rows, int64_t n, int64_t k) {
  double unsplit = -1.0;
  double split = -1.0;
  for (const StepTile &tile : kStepTiles) {
    for (const int64_t splits : kStepSplits) {
      const double us = step_split_us(tile, rows, n, k, splits);
      double &least = splits > 1 ? split : unsplit;
      least = us >= 0.0 && (least < 0.0 || us < least) ? us : least;
    }
  }
  return split >= 0.0 && split <= unsplit;
}

GemmChoice choose_step_tile(const GemmChoice &base, int64_t rows, int64_t n, int64_t k) {
  const int64_t slabs = (k + 63) / 64;
  GemmChoice best = base;
  const double base_us = step_us(base, rows, n, k, 1.0);  // a column split's lower price
  if (base_us < 0.0) {
    return base;
  }
  double best_us = base_us * (1.0 - kStepGain);
  const double stream = 2.0 * static_cast<double>(n) * static_cast<double>(k) / kStepWeightBytesPerUs;
  for (const StepTile &tile : kStepTiles) {
    for (const int64_t splits : kStepSplits) {
      const double us = step_split_us(tile, rows, n, k, splits);
      if (us >= 0.0 && us < best_us) {
        best = {GemmKind::Tile, tile.variant, splits > 1 ? (slabs + splits - 1) / splits * 64 : k, splits};
        best_us = us;
      }
    }
    // A first launch of nearly whole rounds, and the remaining columns in a second one.
    const TileShape &shape = kTileShapes[tile.variant];
    const int64_t token_tiles = (rows + shape.bm - 1) / shape.bm;
    for (int64_t rounds = 1; kComputeUnits * rounds / token_tiles * shape.bn < n; ++rounds) {
      const int64_t weight_tiles = kComputeUnits * rounds / token_tiles;
      const int64_t idle = kComputeUnits * rounds - token_tiles * weight_tiles;
      if (weight_tiles == 0 || idle * 12 > kComputeUnits) {
        continue;
      }
      const int64_t n1 = weight_tiles * shape.bn;
      const double first = kStepLaunchUs + stream + step_compute_us(tile, rows, n1, slabs, 1);
      if (kStepTailScale * first + kStepTailUs >= best_us) {
        break;  // and so do more rounds of this shape
      }
      for (const StepTile &other : kStepTiles) {
        const double us = kStepTailScale * (first + step_compute_us(other, rows, n - n1, slabs, 1)) + kStepTailUs;
        if (us < best_us) {
          best = {GemmKind::Tile, tile.variant, k, 1};
          best.tail_variant = other.variant;
          best.tail_columns = n - n1;
          best_us = us;
        }
      }
    }
  }
  return best;
}

// The fused gather's prologue (slot list, full-row sums of squares, staging) runs in every
// workgroup, so the fused gate_up takes the fewest K slices that fit LDS (measured: 4
// slices of Qwen3-8B gate_up took 47 + 5 us against 38 us for one).  Up to kSplitMaxRows
// rows the split kernel can fuse the gather as well: each workgroup stages the rows' whole
// K (at most kSplitGatherMaxK columns) while its first weight chunks are in flight, which
// the model prices at kSplitGatherRoundUs per round of workgroups over the plain split
// kernel; for projections of many units, split_gathered_kernel gathers once per workgroup
// of a two-per-CU persistent grid instead.
GemmChoice choose_dense_gate_up(int64_t capacity, int64_t n, int64_t k, bool &fused) {
  // 9 to 16 rows: the resident kernel with the gather fused, wherever one part covers K.
  // Measured on MI355X (kernel durations at 9 / 16 rows, weights streamed from HBM) against
  // the choices of the decode models: Qwen3-8B 40.0 / 40.0 us (stream kernel, gather fused)
  // -> 37.9 / 38.9, Qwen3-4B 28.0 / 28.6 (the same) -> 24.0 / 24.7, Qwen3-1.7B 4.5 + 17.3 /
  // 4.6 + 19.0 (gather launch, split kernel) -> 17.1 / 17.8, Qwen3-0.6B 3.1 + 8.7 / 3.5 + 9.5
  // -> 10.0 / 10.4.
  double resident_us = 0.0;
  const GemmChoice resident = choose_resident(capacity, n, k, true, resident_us);
  if (resident_us >= 0.0) {
    fused = true;
    return resident;
  }
  fused = capacity <= kDecodeMaxRows && n * k * 2 <= INT32_MAX;
  if (!fused) {
    return choose_gemm(capacity, n, k, true);
  }
  GemmChoice fused_choice{GemmKind::Stream, 0, 0, 1};
  for (int64_t slices = 1;; ++slices) {
    const int64_t k_slice = ((k + slices - 1) / slices + kStreamSliceQuantum - 1) / kStreamSliceQuantum *
                            kStreamSliceQuantum;
    if (kStreamTokens * (k_slice + kStreamRowPad) * 2 <= kStreamLdsBytes) {
      fused_choice.k_slice = k_slice;
      break;
    }
  }
  // The fused launch streams the weights with one workgroup per 8 weight-row blocks (and K
  // slice); a separate gather launch lets the split kernel spread a small projection over
  // more workgroups (Qwen3-0.6B gate_up at one row: 48 fused workgroups, 13.6 us).
  const int64_t groups = ((n + 15) / 16 + kStreamWaves - 1) / kStreamWaves;
  const int64_t slices = stream_slices(k, fused_choice.k_slice);
  double fused_us = decode_stream_us(n, k, slices * groups, kStreamWorkgroupBytesPerUs, kStreamBytesPerUs,
                                     kStreamFixedUs) +
                    kStreamGatherUs * static_cast<double>((slices * groups + kComputeUnits - 1) / kComputeUnits);
  if (slices > 1) {
    fused_us += kStreamReduceUs + 8.0 * static_cast<double>(slices * capacity * n) / kStreamPartialBytesPerUs;
  }
  double separate_us = 0.0;
  const GemmChoice separate = choose_decode(capacity, n, k, separate_us);
  if (capacity <= kSplitGroupTokens && k <= kSplitGatherMaxK) {
    double split_us = 0.0;
    const GemmChoice split = choose_split(capacity, n, k, split_us, true);
    // The persistent variant prices as the split kernel at one row (its token pieces come
    // from LDS) plus its gather round trip, when the projection has units for every slot.
    // A reduction length of at most 128 has no K range of two chunks: choose_split then finds
    // no persistent split (k_slice 0, cost -1) and the persistent kernel is not a candidate.
    double persistent_us = 0.0;
    GemmChoice persistent = choose_split(1, n, k, persistent_us, false, true);
    const bool persistent_found = persistent.k_slice > 0 && persistent_us >= 0.0;
    persistent_us += kSplitPersistentGatherUs;
    const int64_t units = ((n + 15) / 16 * persistent.k_split + kSplitWaves - 1) / kSplitWaves;
    if (persistent_found && units >= kSplitGatheredWorkgroups && persistent_us < fused_us &&
        persistent_us < split_us && persistent_us < kGatherUs + separate_us) {
      persistent.kind = GemmKind::SplitGathered;
      return persistent;
    }
    if (split_us < fused_us && split_us <= kGatherUs + separate_us) {
      return split;  // fused into the split kernel
    }
  }
  if (kGatherUs + separate_us < fused_us) {
    fused = false;
    return separate;
  }
  return fused_choice;
}

GemmChoice refine_dense_choice(const GemmChoice &base, int64_t rows, int64_t n, int64_t k) {
  return base.kind == GemmKind::Tile && rows >= kStepMinRows ? choose_step_tile(base, rows, n, k) : base;
}

size_t refined_scratch_bytes(int64_t capacity, int64_t n, int64_t k) {
  // A column split keeps no sums, so where neither choice splits K without one, neither does
  // with one; pricing those is most of a choice's host time at many rows.
  const GemmChoice whole = choose_gemm(capacity, n, k, false, false);
  if (whole.kind == GemmKind::Tile && whole.k_split == 1 &&
      (capacity < kStepMinRows || !step_split_pays(capacity, n, k))) {
    return 0;
  }
  return gemm_scratch_bytes(refine_dense_choice(choose_gemm(capacity, n, k, false), capacity, n, k), capacity, n, k);
}

// The tile and K split of a biased projection at `rows` rows (unsplit when `scratch_bytes` has no
// room for the ranges' sums), and its modelled time.
GemmChoice choose_extended(int64_t rows, int64_t n, int64_t k, size_t scratch_bytes, double &us) {
  const int64_t slabs = (k + 63) / 64;
  GemmChoice best{GemmKind::Tile, 0, k, 1};
  us = -1.0;
  for (int variant = 0; variant < kExtendedTileShapes; ++variant) {
    for (const int64_t splits : kStepSplits) {
      const int64_t per_range = (slabs + splits - 1) / splits;
      if (splits > 1 && (per_range < kStepMinSlabs || (splits - 1) * per_range >= slabs ||
                         static_cast<uint64_t>(splits * rows * n * 4) > scratch_bytes)) {
        continue;
      }
      const GemmChoice choice{GemmKind::Tile, variant, splits > 1 ? per_range * 64 : k, splits};
      const double cost = step_us(choice, rows, n, k);
      if (us < 0.0 || cost < us) {
        best = choice;
        us = cost;
      }
    }
  }
  return best;
}

GemmChoice choose_unsplit(int64_t rows, int64_t n, int64_t k) {
  double us = 0.0;
  // The split kernel adds its K ranges in LDS.
  return rows <= kSplitMaxRows && n * k * 2 <= INT32_MAX ? choose_split(rows, n, k, us)
                                                          : choose_extended(rows, n, k, 0, us);
}

KernelLaunch make_extended_gemm(const GemmArgs &args, int64_t capacity, bool gated, const GemmChoice &choice) {
  if (choice.k_split > 1) {
    return make_gemm(args, capacity, gated, choice).main;  // the ranges' sums
  }
  const TileShape &shape = kTileShapes[choice.variant];
  GemmArgs record = args;
  record.capacity = capacity;
  record.k_slice = choice.k_slice;
  record.k_split = 1;
  KernelLaunch kernel;
  kernel.func = args.payload == kPayloadF16 ? ExtendedKernels<F16Payload>::tile(gated, choice.variant)
                                            : ExtendedKernels<Bf16Payload>::tile(gated, choice.variant);
  kernel.grid = dim3(static_cast<unsigned>((args.n + shape.bn - 1) / shape.bn),
                     static_cast<unsigned>((capacity + shape.bm - 1) / shape.bm), 1);
  kernel.block = dim3(static_cast<unsigned>(64 * shape.waves), 1, 1);
  kernel.set_args(record);
  return kernel;
}

bool split_gather_fusable(int64_t capacity, int64_t n, int64_t k) {
  const GemmChoice choice = choose_gemm(capacity, n, k, false);
  return choice.kind == GemmKind::Split && choice.variant == 1 && k <= kSplitGatherMaxK;
}

// K ranges whose fp32 partial sums go through scratch and the reduction kernel.
int64_t scratch_slices(GemmChoice choice, int64_t k) {
  switch (choice.kind) {
    case GemmKind::Stream:
      return stream_slices(k, choice.k_slice);
    case GemmKind::Tile:
    case GemmKind::Resident:
      return choice.k_split;
    default:
      return 1;  // the split kernel sums its K ranges in LDS
  }
}

size_t gemm_scratch_bytes(GemmChoice choice, int64_t capacity, int64_t n, int64_t k) {
  const int64_t slices = scratch_slices(choice, k);
  if (slices == 1) {
    return 0;
  }
  const size_t partial_bytes = static_cast<size_t>(slices * capacity * n) * sizeof(float);
  return (partial_bytes + 255) / 256 * 256;
}

hipError_t enable_large_lds(const void *func) {
  // (function, device) pairs already opted in: a few stream kernels on a few devices, kept in
  // a fixed table so that no launch path allocates.  Past its end the attribute is set again
  // on every launch (harmless, only slower).
  struct Enabled {
    const void *func;
    int device;
  };
  static std::mutex mutex;
  static Enabled enabled[128];
  static int count = 0;
  int device = 0;
  if (const hipError_t status = hipGetDevice(&device); status != hipSuccess) {
    return status;
  }
  std::lock_guard<std::mutex> guard(mutex);
  for (int index = 0; index < count; ++index) {
    if (enabled[index].func == func && enabled[index].device == device) {
      return hipSuccess;
    }
  }
  // The dynamic maximum is what the CU's 160 KB leave beside the function's static LDS (the
  // split kernel's partial sums, the fused gather's row table).
  hipFuncAttributes attributes{};
  if (const hipError_t status = hipFuncGetAttributes(&attributes, func); status != hipSuccess) {
    return status;
  }
  const int limit = 160 * 1024 - static_cast<int>(attributes.sharedSizeBytes);
  const hipError_t status = hipFuncSetAttribute(func, hipFuncAttributeMaxDynamicSharedMemorySize, limit);
  if (status == hipSuccess && count < static_cast<int>(sizeof(enabled) / sizeof(enabled[0]))) {
    enabled[count++] = Enabled{func, device};
  }
  return status;
}

GemmLaunch make_gemm(const GemmArgs &args, int64_t capacity, bool gated, GemmChoice choice, bool fused_gather) {
  GemmLaunch launches;
  KernelLaunch &kernel = launches.main;
  const bool f16 = args.payload == kPayloadF16;
  auto tile_kernel = [&](int variant) {
    const WeightLoads loads = capacity > kTileShapes[variant].bm ? WeightLoads::Shared
                              : args.k % kRotatedPitch == 0 && choice.k_split <= kRotatedRanges
                                  ? WeightLoads::StreamRotated
                                  : WeightLoads::Stream;
    return f16 ? DenseKernels<F16Payload>::tile(gated, variant, loads) : DenseKernels<Bf16Payload>::tile(gated, variant, loads);
  };
  GemmArgs record = args;
  record.capacity = capacity;
  record.k_slice = choice.k_slice;
  record.k_split = choice.k_split;
  if ((choice.kind == GemmKind::Split || choice.kind == GemmKind::SplitGathered) &&
      (choice.k_slice <= 0 || choice.k_split <= 0)) {
    launches.usable = false;  // an empty K range would read nothing and store zeros
    return launches;
  }
  if (choice.kind == GemmKind::Split) {
    // choose_split is only consulted up to kSplitMaxRows rows (and the fused gather up to
    // one token group).
    const int64_t per_group = kSplitWaves / choice.k_split;
    // 8-row weight blocks while 16-row ones would fill at most half the CUs.
    const bool half = ((args.n + 15) / 16 + per_group - 1) / per_group * 2 <= kComputeUnits;
    const int64_t row_blocks = half ? (args.n + 7) / 8 : (args.n + 15) / 16;
    // The gather fuses into one token group (gate_up of a Dense step, the MoE router).
    const bool gather = fused_gather && choice.variant == 1;
    kernel.func = f16 ? DenseKernels<F16Payload>::split(gated, choice.variant, gather, half)
                      : DenseKernels<Bf16Payload>::split(gated, choice.variant, gather, half);
    kernel.grid = dim3(static_cast<unsigned>((row_blocks + per_group - 1) / per_group), 1, 1);
    kernel.block = dim3(64 * kSplitWaves, 1, 1);
    // Dynamic LDS beyond 64 KB: launch() opts the function in (enable_large_lds).
    kernel.shmem = gather ? static_cast<unsigned>(
                                (capacity < kSplitGroupTokens ? capacity : kSplitGroupTokens) * (args.k + 16) * 2)
                          : 0u;
  } else if (choice.kind == GemmKind::SplitGathered) {
    // Chosen only for a Dense step's gate_up with the gather fused.
    const int64_t row_blocks = (args.n + 15) / 16;
    const int64_t units = (row_blocks * choice.k_split + kSplitWaves - 1) / kSplitWaves;
    kernel.func = f16 ? DenseKernels<F16Payload>::split_gathered(gated) : DenseKernels<Bf16Payload>::split_gathered(gated);
    kernel.grid = dim3(static_cast<unsigned>(units < kSplitGatheredWorkgroups ? units : kSplitGatheredWorkgroups), 1, 1);
    kernel.block = dim3(64 * kSplitWaves, 1, 1);
    kernel.shmem = static_cast<unsigned>((capacity < kSplitGroupTokens ? capacity : kSplitGroupTokens) * (args.k + 16) * 2 +
                                         kSplitGatheredScratchBytes);
  } else if (choice.kind == GemmKind::Resident) {
    const int64_t row_blocks = (args.n + 15) / 16;
    const int cpw = static_cast<int>(choice.k_slice / (kResidentWaves * kResidentChunk));
    const int64_t walkers = std::min<int64_t>(kResidentWorkgroups / choice.k_split, row_blocks);
    kernel.func = f16 ? DenseKernels<F16Payload>::resident(gated, fused_gather && gated, cpw, choice.variant)
                      : DenseKernels<Bf16Payload>::resident(gated, fused_gather && gated, cpw, choice.variant);
    if (kernel.func == nullptr) {
      launches.usable = false;
      return launches;
    }
    kernel.grid = dim3(static_cast<unsigned>(choice.k_split * walkers), 1, 1);
    kernel.block = dim3(64 * kResidentWaves, 1, 1);
  } else if (choice.kind == GemmKind::Stream) {
    const int64_t groups = ((args.n + 15) / 16 + kStreamWaves - 1) / kStreamWaves;
    const int64_t slices = stream_slices(args.k, choice.k_slice);
    const bool gather = fused_gather && gated;
    kernel.func = f16 ? DenseKernels<F16Payload>::stream(gated, gather) : DenseKernels<Bf16Payload>::stream(gated, gather);
    kernel.grid = dim3(static_cast<unsigned>(slices * groups), 1, 1);
    kernel.block = dim3(64 * kStreamWaves, 1, 1);
    // Dynamic LDS beyond 64 KB: launch() opts the function in (enable_large_lds).
    kernel.shmem = static_cast<unsigned>(kStreamTokens * (choice.k_slice + kStreamRowPad) * 2);
  } else {
    // Tile grid over weight rows [0, n1) (all of them without a column split); the tail
    // launch takes [n1, n): its weights, and its output columns (half as many for gate_up).
    const int64_t n1 = args.n - choice.tail_columns;
    if (choice.tail_columns > 0) {
      if (choice.k_split != 1 || choice.tail_variant < 0 || n1 <= 0 || (gated && n1 % 2 != 0)) {
        launches.usable = false;
        return launches;
      }
      record.n = n1;
      const TileShape &other = kTileShapes[choice.tail_variant];
      GemmArgs tail_record = record;
      tail_record.n = choice.tail_columns;
      tail_record.w = args.w + n1 * args.k;
      tail_record.out = args.out + (gated ? n1 / 2 : n1);
      launches.tail.func = tile_kernel(choice.tail_variant);
      launches.tail.grid = dim3(static_cast<unsigned>((tail_record.n + other.bn - 1) / other.bn),
                                static_cast<unsigned>((capacity + other.bm - 1) / other.bm), 1);
      launches.tail.block = dim3(static_cast<unsigned>(64 * other.waves), 1, 1);
      launches.tail.set_args(tail_record);
    }
    const TileShape &shape = kTileShapes[choice.variant];
    kernel.func = tile_kernel(choice.variant);
    kernel.grid = dim3(static_cast<unsigned>((n1 + shape.bn - 1) / shape.bn),
                       static_cast<unsigned>((capacity + shape.bm - 1) / shape.bm),
                       static_cast<unsigned>(choice.k_split));
    kernel.block = dim3(static_cast<unsigned>(64 * shape.waves), 1, 1);
  }
  if (scratch_slices(choice, args.k) > 1) {
    launches.slices = scratch_slices(choice, args.k);
    KernelLaunch &reduce = launches.reduce;
    reduce.func = f16 ? DenseKernels<F16Payload>::stream_reduce(gated) : DenseKernels<Bf16Payload>::stream_reduce(gated);
    reduce.grid = dim3(static_cast<unsigned>((capacity * (args.n / 4) + 255) / 256), 1, 1);
    reduce.block = dim3(256, 1, 1);
    reduce.set_args(record);
  }
  kernel.set_args(record);
  return launches;
}

// Grouped projections run on the tile kernel's grouped instantiations, one per expert
// tile height (choose_moe_tile picks it by routes per expert): 64 x 128 (four waves, three
// stages, 72 KB of LDS: two workgroups per CU), 128 x 256 (eight waves, three stages,
// nontemporal or plain weight loads) and 256 x 128 (eight waves, three stages, nontemporal),
// the last two at 144-147 KB of LDS, one workgroup per CU.  With few routes per expert a
// tile's K loop is short against its prologue and epilogue, and the second workgroup of a
// CU streams while the first fills or drains (Qwen3-30B-A3B layer at 256 / 512 tokens:
// 281 / 294 us on a 64 x 256 eight-wave tile with four stages, one per CU, against 255 /
// 265 us).  The nontemporal hint suits tiles whose expert's weights no other tile reads;
// with plain loads an expert split over two 128-row tiles reads its weights from the
// last-level cache the second time.
struct GroupedTile {
  int bm;
  int bn;
  int waves;
};

// The down projection (not gated) of the 128-row regimes takes 128 x 128 tiles of two
// stages (64 KB of LDS, two workgroups per CU): its K loop is short (Qwen3-30B-A3B: 768
// columns, 12 slabs), so a tile's fill and drain weigh on it, and the CU's second workgroup
// streams meanwhile.  Measured on that layer against 128 x 256 three-stage down tiles:
// 600 / 800 / 1024 tokens 306.8 / 311.6 / 319.6 -> 301.3 / 306.0 / 314.6 us, 1100 / 1400 /
// 1700 / 2048 tokens 346.3 / 350.2 / 385.1 / 396.4 -> 338.7 / 343.2 / 379.1 / 389.9 us.
// gate_up (K = 2048) lost on such tiles (2048 tokens: 410-421 against 397 us).
GroupedTile grouped_tile(MoeTile tile, bool gated) {
  switch (tile) {
    case MoeTile::Rows64:
      return {64, 128, 4};
    case MoeTile::Rows128Stream:
    case MoeTile::Rows128:
      return gated ? GroupedTile{128, 256, 8} : GroupedTile{128, 128, 8};
    case MoeTile::Rows256:
      return {256, 128, 8};
    default:
      return {0, 0, 0};
  }
}

int grouped_tile_rows(MoeTile tile) { return grouped_tile(tile, true).bm; }  // the same for down

KernelLaunch make_grouped_gemm(const GemmArgs &args, bool gated, int max_tiles, MoeTile tile) {
  const GroupedTile shape = grouped_tile(tile, gated);
  const bool extended =
      args.bias != nullptr || args.act.function == kActivationRelu || args.act.function == kActivationGelu;
  const void *func = args.payload == kPayloadF16 ? GroupedKernels<F16Payload>::tile(gated, tile, extended)
                                                 : GroupedKernels<Bf16Payload>::tile(gated, tile, extended);
  if (max_tiles % 8 != 0 || func == nullptr) {
    return KernelLaunch{};  // grouped_tile_coordinates needs a multiple of 8 (callers pad)
  }
  GemmArgs record = args;
  record.k_slice = args.k;
  record.k_split = 1;
  record.partials = nullptr;
  KernelLaunch kernel;
  kernel.func = func;
  kernel.grid = dim3(static_cast<unsigned>((args.n + shape.bn - 1) / shape.bn), static_cast<unsigned>(max_tiles), 1);
  kernel.block = dim3(static_cast<unsigned>(64 * shape.waves), 1, 1);
  kernel.set_args(record);
  return kernel;
}

// Routes per expert tile of the grouped split kernel: one 16-column MFMA token block.
int grouped_split_rows() { return 16; }

// K ranges per weight block: two (both waves of a workgroup on one block) where each still has
// at least four 128-wide chunks.  Every pairing of 1 to 8 ranges with 1 to 8 waves, forced on the
// Qwen3-30B-A3B layer and a 1024 x 512, 64-expert one at 1 to 64 tokens: this is the fastest or
// within 2 % of it (gate_up K = 2048 at 32 tokens 185.7 us, one range 190.2; down K = 768 185.7,
// two ranges 193.1).
KernelLaunch make_grouped_split(const GemmArgs &args, bool gated, int max_tiles) {
  const int64_t row_blocks = (args.n + 15) / 16;
  const int64_t chunks = (args.k + 127) / 128;
  const int64_t ksplit = chunks >= 4 * kGroupedSplitWaves ? kGroupedSplitWaves : 1;
  GemmArgs record = args;
  record.k_split = ksplit;
  record.k_slice = (chunks + ksplit - 1) / ksplit * 128;
  record.partials = nullptr;
  KernelLaunch kernel;
  kernel.func = args.payload == kPayloadF16 ? GroupedKernels<F16Payload>::split(gated)
                                            : GroupedKernels<Bf16Payload>::split(gated);
  kernel.grid = dim3(static_cast<unsigned>((row_blocks * ksplit + kGroupedSplitWaves - 1) / kGroupedSplitWaves),
                     static_cast<unsigned>(max_tiles), 1);
  kernel.block = dim3(64 * kGroupedSplitWaves, 1, 1);
  kernel.set_args(record);
  return kernel;
}

std::string gemm_name(GemmChoice choice, bool gated) {
  const std::string prefix = gated ? "_gated" : "";
  if (choice.kind == GemmKind::Split) {
    return "split" + prefix + "_t" + std::to_string(kSplitGroupTokens * choice.variant) + "_k" +
           std::to_string(choice.k_split);
  }
  if (choice.kind == GemmKind::SplitGathered) {
    return "split" + prefix + "_t8_k" + std::to_string(choice.k_split) + "_persistent";
  }
  if (choice.kind == GemmKind::Stream) {
    return "stream" + prefix + "_t16";
  }
  if (choice.kind == GemmKind::Resident) {
    std::string name = "resident" + prefix + "_t" + std::to_string(8 * choice.variant) + "_c" +
                       std::to_string(choice.k_slice / (kResidentWaves * kResidentChunk));
    if (choice.k_split > 1) {
      name += "_p" + std::to_string(choice.k_split);
    }
    return name;
  }
  const TileShape &shape = kTileShapes[choice.variant];
  std::string name = "tile" + prefix + "_" + std::to_string(shape.bm) + "x" + std::to_string(shape.bn);
  if (choice.k_split > 1) {
    name += "_k" + std::to_string(choice.k_split);
  }
  if (choice.tail_columns > 0) {
    const TileShape &other = kTileShapes[choice.tail_variant];
    name += "+" + std::to_string(other.bm) + "x" + std::to_string(other.bn) + "_n" + std::to_string(choice.tail_columns);
  }
  return name;
}

}  // namespace xp
