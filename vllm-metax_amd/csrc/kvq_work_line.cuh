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

// a / b, both >= 0.  A 64-bit division is a routine of over a hundred instructions, at 2.4 ns each for a wave alone on its SIMD,
// as in a launch's prologue and its reduce; a line of up to 16 million units on 256 workgroups takes the short one.  With it, the
// prologue that holds the lengths and the reduce's notes, a step of 200 sequences (4 kv heads, int4 codes) went 42.9 -> 40.0 us,
// of 250 short ones on 8 kv heads 37.5 -> 33.3, of 20 35.0 -> 34.2.
__device__ __forceinline__ int64_t line_div(int64_t a, int64_t b) {
  return (((uint64_t)a | (uint64_t)b) >> 32) == 0 ? (int64_t)((uint32_t)a / (uint32_t)b) : a / b;
}

// A line of units is shared out over at most as many workgroups as it has units (active_workgroups, and the batch-invariant
// line's own count), so no share of a line that is not empty is empty; the reduces rely on it.
__device__ __forceinline__ int64_t wg_tile_begin(int w, int64_t total, int num_wg) {
  return line_div((int64_t)w * total, num_wg);
}

// The workgroup that holds unit x: the largest w with wg_tile_begin(w) <= x.
__device__ __forceinline__ int wg_of_unit(int64_t x, int64_t total, int num_wg) {
  return (int)line_div((x + 1) * num_wg - 1, total);
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
