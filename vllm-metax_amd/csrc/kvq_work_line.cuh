// How the balanced split-K launches ("stream-K") cut their line of tiles into the workgroups' shares.
#pragma once

#include "kvq_internal.h"

namespace kvq {

// Starting on a sequence (query row, first tile with nothing in flight, folding and storing the state of the
// one before) costs a workgroup 4 - 5 us, whatever the number of kv heads it serves; the work line that is cut into
// equal shares therefore charges every sequence StreamKArgs::setup_units units before its tiles.  A unit is a
// tile of the workgroup's run, and the 8 / HPW waves of a head take a run's tiles in turn, so a unit lasts
// 2.9 us / (8 / HPW) and the charge grows with the waves per head (setup_units_for).  Measured on MI355X at batch 64,
// 1k..8k tokens: with eight kv heads and no charge, workgroups whose share crossed a sequence boundary ran 2.9 us
// (one tile time) longer than the others and were the last to finish; with one kv head and a charge of one unit
// they ran 23.0 us against 18.2 us and the launch waited for them.
constexpr int setup_units_for(int waves_per_head) { return waves_per_head == 1 ? 1 : 3 * waves_per_head / 2; }

__device__ __forceinline__ int64_t wg_tile_begin(int w, int64_t total, int num_wg) {
  return ((int64_t)w * total) / num_wg;
}

// Workgroups that take a share of a line of `total` units: all that were launched, unless the line
// is so short that a share would fall below kMinUnitsPerWg -- a small batch is then spread over
// fewer workgroups, so that a sequence is not cut into dozens of one-tile partial states for the
// reduce to merge.  Measured at batch 4 x 512 tokens (main + reduce kernel): 15.6 us with shares of
// at least 2 units, 18.3 us with 4 (a tile at a time per wave: about 4 us per tile at low load).
constexpr int kMinUnitsPerWg = 2;
__device__ __forceinline__ int active_workgroups(int64_t total, int num_wg) {
  const int64_t want = total / kMinUnitsPerWg;
  return want >= num_wg ? num_wg : (want < 1 ? 1 : (int)want);
}

}  // namespace kvq
