// Device code and launch templates of the paged decode kernels, instantiated once per head size and query type in
// kvq_paged_decode_d<head size>_<type>.hip (one translation unit each, so they compile in parallel).
#pragma once

#include <type_traits>

#include "kvq_attn_core.cuh"
#include "kvq_work_line.cuh"

namespace kvq {

int heads_per_wg(int num_kv_heads);

// Tiles of a decode sequence of `len` > 0 tokens: those that hold a token of the row's window,
// [window_first / 32, ceil(len / 32)).
__device__ __forceinline__ int decode_tiles(int len, int window) {
  return (len + kTile - 1) / kTile - window_first(len, window) / kTile;
}

// A sequence's length and its query rows [q0, q1).
struct SeqRow {
  int len, q0, q1;
};
__device__ __forceinline__ SeqRow load_seq(const StreamKArgs& a, int s) {
  SeqRow r;
  r.len = a.seq_lens[s];
  r.q0 = a.cu_seqlens_q != nullptr ? a.cu_seqlens_q[s] : s;
  r.q1 = a.cu_seqlens_q != nullptr ? a.cu_seqlens_q[s + 1] : s + 1;
  return r;
}
// Its tiles as a decode sequence: 0 for query runs and empty ones (the former are the prefill kernels').
__device__ __forceinline__ int seq_tiles(const SeqRow& r, int window) {
  return r.q1 - r.q0 == 1 && r.len > 0 ? decode_tiles(r.len, window) : 0;
}

// Batch-invariant cutting (StreamKArgs::fixed_spans): a sequence is cut at places that depend on nothing but its
// own length -- into at most kFixedSpans spans of equal size, none shorter than kMinSpanTiles tiles.  The spans of
// all decode sequences form one line (a unit per span) that is cut into equal shares like the balanced line, so
// WHICH workgroup computes a span depends on the batch, but not what it computes: the states of a sequence's
// spans lie in slots seq * kFixedSpans + span and are merged in span order, so a row's bits are the same
// whatever else the batch holds and however many workgroups the device runs.
constexpr int kFixedSpans = 32;
constexpr int kMinSpanTiles = 8;
__device__ __forceinline__ int fixed_span_tiles(int ntiles) {
  const int per = (ntiles + kFixedSpans - 1) / kFixedSpans;
  return per > kMinSpanTiles ? per : kMinSpanTiles;
}
__device__ __forceinline__ int fixed_span_count(int ntiles) {
  const int per = fixed_span_tiles(ntiles);
  return (ntiles + per - 1) / per;   // 0 for no tiles
}

// Units of a sequence on the line the launch cuts: its setup charge, then one per tile, or (FIXED) its spans.
template <bool FIXED>
__device__ __forceinline__ int seq_line_units(const SeqRow& r, int window, int setup) {
  const int n = seq_tiles(r, window);
  if constexpr (FIXED) return fixed_span_count(n);
  else return n > 0 ? n + setup : 0;
}

// The same for sequence s, 0 past the last.  No branch on it: a lane past the last sequence rereads the last one and drops
// the result, so that the loads of a lane's chunks all go out together.
template <bool FIXED>
__device__ __forceinline__ int line_units(const StreamKArgs& a, int s) {
  const int n = seq_line_units<FIXED>(load_seq(a, min(s, a.num_seqs - 1)), a.io.window, a.setup_units);
  return s < a.num_seqs ? n : 0;
}

// The scans over more than 64 sequences work on chunks of 64 (one per lane), kScanBatch chunks per step so that their
// loads are in flight together (batch 512: 16 dependent round trips -> 4).
constexpr int kScanBatch = 4;

// Total units of the work line.
template <bool FIXED>
__device__ __forceinline__ int64_t scan_total(const StreamKArgs& a, int lane) {
  const int B = a.num_seqs;
  int64_t total = 0;
  for (int base = 0; base < B; base += kWave * kScanBatch) {
    int n[kScanBatch];
#pragma unroll
    for (int j = 0; j < kScanBatch; ++j)
      n[j] = line_units<FIXED>(a, base + kWave * j + lane);
#pragma unroll
    for (int j = 0; j < kScanBatch; ++j) total += __builtin_amdgcn_readlane(wave_incl_scan(n[j]), 63);
  }
  return total;
}

// The sequence that holds unit `lo` and the index of its first unit.
template <bool FIXED>
__device__ __forceinline__ void scan_locate(const StreamKArgs& a, int lane, int64_t lo, int& seq, int64_t& seq_start) {
  const int B = a.num_seqs;
  int64_t cum = 0;
  bool found = false;
  for (int base = 0; base < B && !found; base += kWave * kScanBatch) {
    int nn[kScanBatch];
#pragma unroll
    for (int j = 0; j < kScanBatch; ++j)
      nn[j] = line_units<FIXED>(a, base + kWave * j + lane);
#pragma unroll
    for (int j = 0; j < kScanBatch; ++j) {
      const int n = nn[j];
      const int incl = wave_incl_scan(n);
      const int64_t first = cum + incl - n, last = cum + incl;
      const uint64_t hit = __builtin_amdgcn_ballot_w64(n > 0 && first <= lo && lo < last);
      if (hit != 0 && !found) {
        const int src = __builtin_ctzll(hit);
        seq = base + kWave * j + src;
        seq_start = cum + __builtin_amdgcn_readlane(incl - n, src);
        found = true;
      }
      cum += __builtin_amdgcn_readlane(incl, 63);
    }
  }
}

// HPW = kv heads per workgroup (1, 2, 4 or 8).  A workgroup always has eight waves: with fewer than
// eight kv heads the 8 / HPW waves of a head take the tiles of a run in turn and their states are
// folded together in LDS when the run ends, so a compute unit keeps eight tile streams in flight
// whatever the head count and a sequence is cut into no more partial states than with eight heads.
// FIXED: the batch-invariant cutting instead of the balanced one (a template argument, so that the balanced
// kernel carries none of it: as a run-time branch it cost the headline launch 0.6 us).
template <int D, int QDT, int HPW, bool CAP, int CODE, bool STREAM, bool FIXED = false>
__global__ __launch_bounds__(512) void paged_decode_streamk_kernel(StreamKArgs a) {
  using DTile = DecodeTile<D, QDT, kRuntimeDtype, CODE, STREAM>;
  constexpr int NSUB = 8 / HPW;
  __shared__ __align__(16) uint8_t lds[8][DTile::LDS_WAVE];
  const int lane = threadIdx.x & 63;
  // Uniform to the compiler as well: with several waves per kv head the tile number follows from the wave's, and as a
  // vector value it turned every tile load into a loop over the lanes' descriptors and the block-table reads into
  // vector loads, whose wait drained the tile in flight (200 sequences of 60-2000 tokens, int4 cache, 4 kv heads: a
  // step 50.9 -> 45.5 us).
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sub = wave % NSUB;
  const int hkv = blockIdx.y * HPW + wave / NSUB;
  if (hkv >= a.io.g.num_kv_heads) return;  // a finished wave no longer counts at the workgroup's barriers
  const int w = blockIdx.x;
  const int B = a.num_seqs;

  constexpr bool fixed = FIXED;

  const LaneOffsets off = DTile::lane_offsets(a.io.g, lane);   // (while the lengths are on their way)

  // the balanced cutting: total units of the work line (each wave redoes this tiny scan; no LDS, no barrier)
  int64_t total = 0, lo = 0, hi = 0;
  int num_wg = 0;
  int seq = 0;
  int64_t seq_start = 0;  // global index of the sequence's first unit
  SeqRow cur{};           // the sequence's length and row
  auto take_share = [&]() __attribute__((always_inline)) {
    // (the batch-invariant line is short -- a unit is a span of at least kMinSpanTiles tiles -- and is always shared
    // out over every workgroup there is a unit for)
    num_wg = fixed ? (total < a.num_wg ? (total < 1 ? 1 : (int)total) : a.num_wg) : active_workgroups(total, a.num_wg);
    if (w >= num_wg) return false;
    lo = wg_tile_begin(w, total, num_wg);
    hi = wg_tile_begin(w + 1, total, num_wg);
    if (lo >= hi) {   // an empty work line: workgroup 0 still reports its length
      if (!fixed && w == 0 && blockIdx.y == 0 && wave == 0 && lane == 0) a.wg_info[0] = total;
      return false;
    }
    return true;
  };
  // Up to 64 N sequences: each lane keeps N of them, and one trip to memory serves the total, the place of the share and
  // the sequence it begins in (200 sequences, 4 kv heads, int4 codes: the three trips one after another cost a step 1 us).
  auto scan_held = [&](auto n_tag) __attribute__((always_inline)) {
    constexpr int N = decltype(n_tag)::value;
    SeqRow mine[N];
    int n[N], incl[N], sum = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) mine[j] = load_seq(a, min(kWave * j + lane, B - 1));
#pragma unroll
    for (int j = 0; j < N; ++j) {
      n[j] = kWave * j + lane < B ? seq_line_units<fixed>(mine[j], a.io.window, a.setup_units) : 0;
      incl[j] = wave_incl_scan(n[j]) + sum;
      sum = __builtin_amdgcn_readlane(incl[j], 63);
    }
    total = sum;
    if (!take_share()) return false;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const uint64_t hit = __builtin_amdgcn_ballot_w64(n[j] > 0 && incl[j] - n[j] <= lo && lo < incl[j]);
      if (N == 1 || hit != 0) {   // (lo < total: there is one)
        const int src = __builtin_ctzll(hit);
        seq = kWave * j + src;
        seq_start = __builtin_amdgcn_readlane(incl[j] - n[j], src);
        cur = {__builtin_amdgcn_readlane(mine[j].len, src), __builtin_amdgcn_readlane(mine[j].q0, src),
               __builtin_amdgcn_readlane(mine[j].q1, src)};
      }
    }
    return true;
  };
  if (B <= kWave) {
    if (!scan_held(std::integral_constant<int, 1>{})) return;
  } else if (B <= kWave * kScanBatch) {
    if (!scan_held(std::integral_constant<int, kScanBatch>{})) return;
  } else {
    total = scan_total<fixed>(a, lane);
    if (!take_share()) return;
    scan_locate<fixed>(a, lane, lo, seq, seq_start);
    seq = __builtin_amdgcn_readfirstlane(seq);
    cur = load_seq(a, seq);
  }
  // Where the share begins (the reduce kernel's key to the span): noted in the first round of the loop, stored
  // after the last.  A store ahead of the tile loads would sit before them in the wave's in-order memory
  // counter, and the first tile would wait for the store's acknowledgement (measured: 0.6 us per launch).
  int info_seq = -1, info_row = 0, info_tiles = 0;
  int64_t info_start = 0;

  // One run of tiles [t_begin, t_end) of sequence `cur` (ntiles tiles from tile t0 on), its state to `slot` unless
  // the run is the whole sequence.
  auto process = [&](int cur, int64_t cur_start, int64_t row, int len, int first, int t0, int ntiles, int t_begin,
                     int t_end, int64_t slot) __attribute__((always_inline)) {
    if (a.k_new != nullptr && t_end == t0 + ntiles) {   // uniform over the workgroup: the run holds the last tile
      const bool padding = a.new_slots != nullptr && a.new_slots[row] < 0;   // uniform: a scalar load
      if (sub == 0 && !padding) write_new_token<D>(a, cur, row, len, hkv, lane);
      // the record is in memory before any wave of the workgroup loads the tile that holds it
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if constexpr (NSUB > 1) lds_barrier();
    }
    typename DTile::State st;
    DTile::template run<CAP>(a.io, off, cur, row, len, first, t_begin, t_end, hkv, lane, lds[wave], st, sub, NSUB);
    // the run holds the sequence's first tile: its place on the line, for the reduce kernel (behind the run's loads)
    if (!fixed && t_begin == t0 && blockIdx.y == 0 && wave == 0 && lane == 0) a.seq_first_unit[cur] = cur_start;
    if constexpr (NSUB > 1) {
      if (sub != 0) DTile::dump_state(st, lane, lds[wave]);
      lds_barrier();
      if (sub == 0) {
#pragma unroll
        for (int j = 1; j < NSUB; ++j)
          if (t_begin + j < t_end) DTile::fold_state(st, lane, lds[wave + j]);  // wave j owned a tile
      }
      lds_barrier();  // the windows may be overwritten by the next run
    }
    if (sub == 0) {
      if (t_begin == t0 && t_end == t0 + ntiles) {
        DTile::emit_final(a.io, row, hkv, lane, st);
      } else {
        DTile::emit_partial(a.io, a.part_o, a.part_ml, slot, hkv, lane, st);
      }
    }
  };

  // (batch-invariant cutting, one wave per kv head) `count` consecutive spans of one sequence as ONE run of tiles: the
  // stream goes on across the spans' edges, where DecodeTile::run stores and restarts the state, so a span's state
  // holds the same bits as if it had been computed alone -- without a query reload and a first tile that nothing
  // prefetched per span.
  auto process_spans = [&](int cur, int64_t row, int len, int first, int t0, int ntiles, int t_begin, int t_end, int per,
                           int span) __attribute__((always_inline)) {
    if (a.k_new != nullptr && t_end == t0 + ntiles) {   // uniform over the workgroup: the run holds the last tile
      const bool padding = a.new_slots != nullptr && a.new_slots[row] < 0;
      if (!padding) write_new_token<D>(a, cur, row, len, hkv, lane);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    }
    typename DTile::State st;
    typename DTile::SpanEdges sp{a.part_o, a.part_ml, (int64_t)cur * kFixedSpans + span, per, per};
    DTile::template run<CAP, true>(a.io, off, cur, row, len, first, t_begin, t_end, hkv, lane, lds[wave], st, 0, 1,
                                   &sp);
    DTile::emit_partial(a.io, a.part_o, a.part_ml, sp.slot, hkv, lane, st);
  };

  if constexpr (fixed) {
    // the spans [lo, hi) of the span line, sequence by sequence
    int64_t at = lo;
    while (at < hi && seq < B) {
      const int ntiles = __builtin_amdgcn_readfirstlane(seq_tiles(load_seq(a, seq), a.io.window));
      const int spans = fixed_span_count(ntiles);
      const int span = (int)(at - seq_start);
      if (span >= spans) {   // also: a sequence without tiles
        seq_start += spans;
        ++seq;
        continue;
      }
      const int per = fixed_span_tiles(ntiles);
      const int len = __builtin_amdgcn_readfirstlane(a.seq_lens[seq]);
      const int64_t row = a.cu_seqlens_q ? (int64_t)a.cu_seqlens_q[seq] : (int64_t)seq;
      const int first = window_first(len, a.io.window);
      const int t0 = first / kTile;
      const int t_begin = t0 + span * per;
      if constexpr (NSUB == 1) {
        const int64_t rest = hi - at;
        const int count = rest < spans - span ? (int)rest : spans - span;   // the sequence's spans inside this share
        if (count > 1) {
          process_spans(seq, row, len, first, t0, ntiles, t_begin, min(t0 + ntiles, t_begin + count * per), per, span);
          at += count;
          continue;
        }
      }
      const int t_end = min(t0 + ntiles, t_begin + per);
      process(seq, 0, row, len, first, t0, ntiles, t_begin, t_end, (int64_t)seq * kFixedSpans + span);
      ++at;
    }
    return;
  }

  const int setup = a.setup_units;
  int64_t pos = lo;
  for (; pos < hi && seq < B; ++seq) {
    const SeqRow nxt = load_seq(a, min(seq + 1, B - 1));   // on its way while this sequence's run is computed
    const int ntiles = seq_tiles(cur, a.io.window);
    if (ntiles == 0) {
      cur = nxt;
      continue;
    }
    const int units = ntiles + setup;
    const int len = cur.len;
    const int64_t row = cur.q0;
    if (info_seq < 0) {
      info_seq = seq;
      info_row = cur.q0;
      info_tiles = ntiles;
      info_start = seq_start;
    }
    const int first = window_first(len, a.io.window);  // tokens before it are outside the window
    const int t0 = first / kTile;                      // the sequence's tile line starts at this tile
    // units [pos, min(hi, end of the sequence)) of the line; the first setup_units of a sequence
    // stand for no tile
    const int u_begin = (int)(pos - seq_start);
    const int64_t rem = hi - seq_start;
    const int u_end = rem < units ? (int)rem : units;
    const int t_begin = t0 + (u_begin > setup ? u_begin - setup : 0);
    const int t_end = t0 + u_end - setup;
    const int64_t start = seq_start;
    pos = seq_start + u_end;
    seq_start += units;
    if (t_begin < t_end)  // else: this share ends inside the setup charge and holds no tile
      process(seq, start, row, len, first, t0, ntiles, t_begin, t_end, (int64_t)w + seq);
    cur = nxt;
  }
  if (blockIdx.y == 0 && wave == 0 && lane == 0) {   // this lane leaves the reduce kernel its notes
    if (w == 0) a.wg_info[0] = total;
    if (info_seq >= 0) {
      const uint32_t first = wg_of_unit(info_start + setup, total, num_wg), last = wg_of_unit(info_start + setup + info_tiles - 1, total, num_wg);
      a.wg_info[2 * w + 2] = (int64_t)((uint64_t)(uint32_t)info_row << 32 | (uint32_t)info_seq);
      a.wg_info[2 * w + 3] = (int64_t)((uint64_t)last << 32 | first);
    }
  }
}

// A workgroup per (kv head, sequence): its eight waves take the sequence's tiles in turn, their states meet in LDS and
// the output row is written there and then -- no partial states, no scan of the lengths, no second launch.  For short
// contexts in a batch that leaves the chip room (whole_sequences): such a step is a chain of latencies, of which the
// second launch with its round trips to the partial states was the longest link (one sequence of 337 tokens: a step
// 15.4 -> 11.6 us).  Any length comes out right: a wave goes on until the sequence ends.
template <int D, int QDT, bool CAP, int CODE, bool STREAM>
__global__ __launch_bounds__(512) void paged_decode_whole_kernel(StreamKArgs a) {
  using DTile = DecodeTile<D, QDT, kRuntimeDtype, CODE, STREAM>;
  constexpr int NSUB = 8;
  __shared__ __align__(16) uint8_t lds[NSUB][DTile::LDS_WAVE];
  const int lane = threadIdx.x & 63;
  const int sub = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int hkv = blockIdx.x, seq = blockIdx.y;
  const LaneOffsets off = DTile::lane_offsets(a.io.g, lane);   // (while the length is on its way)
  const SeqRow cur = load_seq(a, seq);
  if (cur.q1 - cur.q0 != 1) return;
  const int64_t row = cur.q0;
  if (cur.len <= 0) {   // empty sequence: defined output (zeros, lse = -inf)
    for (int i = threadIdx.x; i < a.io.group * D; i += kWave * NSUB) {
      const int head = hkv * a.io.group + i / D;
      store_act_rt(a.io.out_dtype, a.io.out, row * a.io.out_stride_t + (int64_t)head * a.io.out_stride_h + i % D, 0.f);
    }
    if (a.io.lse != nullptr && (int)threadIdx.x < a.io.group)
      a.io.lse[row * a.io.num_q_heads + hkv * a.io.group + threadIdx.x] = -INFINITY;
    return;
  }
  if (a.k_new != nullptr) {
    const bool padding = a.new_slots != nullptr && a.new_slots[row] < 0;   // uniform: a scalar load
    if (sub == 0 && !padding) write_new_token<D>(a, seq, row, cur.len, hkv, lane);
    // the record is in memory before any wave of the workgroup loads the tile that holds it
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
  }
  const int first = window_first(cur.len, a.io.window);
  const int t0 = first / kTile, t_end = t0 + decode_tiles(cur.len, a.io.window);
  typename DTile::State st;
  DTile::template run<CAP>(a.io, off, seq, row, cur.len, first, t0, t_end, hkv, lane, lds[sub], st, sub, NSUB);
  if (sub != 0) DTile::dump_state(st, lane, lds[sub]);
  lds_barrier();
  if (sub != 0) return;
#pragma unroll
  for (int j = 1; j < NSUB; ++j)
    if (t0 + j < t_end) DTile::fold_state(st, lane, lds[j]);   // wave j owned a tile
  DTile::emit_final(a.io, row, hkv, lane, st);
}

// The merge of the batch-invariant cutting: grid (num_seqs, ceil(Hq / 4)), a wave per q head, a lane owns D / 64
// dims.  Lane j takes span j's (m, l); the wave agrees on the maximum and the weights; the spans' outputs are added
// in span order.  Empty decode sequences get their defined output here as well.
template <int D>
__global__ __launch_bounds__(256) void paged_decode_fixed_spans_reduce_kernel(StreamKArgs a) {
  constexpr int V = D / 64;
  static_assert(kFixedSpans <= kWave, "one lane per span");
  const int lane = threadIdx.x & 63;
  const int head = blockIdx.y * 4 + (threadIdx.x >> 6);
  const int seq = blockIdx.x;
  const int Hq = a.io.num_q_heads;
  if (head >= Hq) return;
  const int q0 = a.cu_seqlens_q ? a.cu_seqlens_q[seq] : seq;
  const int q1 = a.cu_seqlens_q ? a.cu_seqlens_q[seq + 1] : seq + 1;
  const int len = a.seq_lens[seq];
  if (q1 - q0 != 1) return;
  const int64_t row = q0;
  const int ntiles = len > 0 ? decode_tiles(len, a.io.window) : 0;
  if (ntiles == 0) {  // empty sequence: defined output (zeros, lse = -inf)
    for (int i = 0; i < V; ++i)
      store_act_rt(a.io.out_dtype, a.io.out, row * a.io.out_stride_t + (int64_t)head * a.io.out_stride_h + lane * V + i, 0.f);
    if (a.io.lse != nullptr && lane == 0) a.io.lse[row * Hq + head] = -INFINITY;
    return;
  }
  const int per = fixed_span_tiles(ntiles);
  const int spans = (ntiles + per - 1) / per;
  if (spans == 1) return;  // written directly by the main kernel
  const int64_t slot0 = (int64_t)seq * kFixedSpans;
  const bool live = lane < spans;
  const int64_t mine = slot0 + (live ? lane : spans - 1);
  const float mj_raw = a.part_ml[(mine * Hq + head) * 2 + 0];
  const float lj_raw = a.part_ml[(mine * Hq + head) * 2 + 1];
  const float mj = live ? mj_raw : -INFINITY;
  const float m = wave_max(mj);
  const float ej = live ? __builtin_amdgcn_exp2f(mj - m) : 0.f;
  const float l = wave_sum(live ? lj_raw * ej : 0.f);
  float acc[V];
#pragma unroll
  for (int i = 0; i < V; ++i) acc[i] = 0.f;
  for (int k0 = 0; k0 < spans; k0 += 8) {   // eight spans per trip to memory, added in span order
    float po[8][V];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int64_t sk = slot0 + min(k0 + k, spans - 1);
      const float* p = a.part_o + (sk * Hq + head) * (int64_t)D + lane * V;
#pragma unroll
      for (int i = 0; i < V; ++i) po[k][i] = p[i];
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float wk = k0 + k < spans ? lane_value(ej, k0 + k) : 0.f;
      const uint32_t kk = wk != 0.f ? 0xffffffffu : 0u;
#pragma unroll
      for (int i = 0; i < V; ++i) acc[i] += as_f32(as_u32(po[k][i]) & kk) * wk;
    }
  }
  const float lt = l + sink_term(a.io.sinks, head, m);
  const float inv = 1.0f / lt;
#pragma unroll
  for (int i = 0; i < V; ++i)
    store_act_rt(a.io.out_dtype, a.io.out, row * a.io.out_stride_t + (int64_t)head * a.io.out_stride_h + lane * V + i, acc[i] * inv);
  if (a.io.lse != nullptr && lane == 0) a.io.lse[row * Hq + head] = (m + __builtin_amdgcn_logf(lt)) * kLn2;
}

// The prefill plan of a mixed batch rides on the reduce launch, one more block of it (PLAN: the last of the grid's first row;
// the rest of its column leaves).  As a launch of its own between the two it cost the step 2 - 3 us (30 decode rows beside 4
// runs of 60 - 300 tokens 77.5 us for 74.8, 12 beside 4 of those 37.4 for 34.6, 200 beside 8 of 60 - 100 70.6 for 68.6; in a step of 60
// rows and 4 x 2048 tokens, 473 us, no more than its runs differ).  An instantiation of its own, since a look at a.plan in front of a decode
// step's reduce took 0.2 us of it.
__device__ __forceinline__ bool plan_block(const StreamKArgs& a) {
  if (blockIdx.x + 1 != gridDim.x) return false;
  if (blockIdx.y == 0 && threadIdx.x < kWave) write_prefill_plan(a.seq_lens, a.cu_seqlens_q, a.num_seqs, a.plan);
  return true;
}

// Merge the partial states of every decode sequence that more than one workgroup touched, and give empty decode
// sequences their defined output.  grid (num_wg, ceil(Hq / 16)), with PLAN (num_wg + 1, ...); 4 waves; a wave takes four
// q heads, 16 lanes each, a lane D/16 dims.
// A sequence is cut only where a workgroup's share begins inside it, so the grid runs over the P workgroups of
// the main kernel, not over the sequences: block w looks at the sequence in which share w begins (the main
// kernel left its number, its row and its shares) and merges it if share w is the
// FIRST to begin inside it; a sequence cut several times is thus merged once, and one that is not cut costs a
// block one round trip.  (A grid over the sequences, every wave scanning all sequence lengths for its place on
// the line, took 44 us at 512 sequences; with one q head per wave the P x Hq waves of this grid, 8192 at 32
// heads, did not fit the chip at once and took 11-13 us.)
template <int D, bool PLAN>
__global__ __launch_bounds__(256) void paged_decode_streamk_reduce_kernel(StreamKArgs a) {
  if constexpr (PLAN)
    if (plan_block(a)) return;
  constexpr int V = D / 16;
  const int lane = threadIdx.x & 63;
  const int sub = lane & 15;           // lane within the head's group of 16
  const int grp = lane & 48;           // first lane of that group
  const int Hq = a.io.num_q_heads;
  const int head_raw = (blockIdx.y * 4 + (threadIdx.x >> 6)) * 4 + (lane >> 4);
  const bool head_ok = head_raw < Hq;
  const int head = head_ok ? head_raw : Hq - 1;   // lanes past the last head repeat it and store nothing
  const int w = blockIdx.x;
  const int B = a.num_seqs;
  // the loads that depend on nothing but the arguments go out before the first branch
  const int64_t total = a.wg_info[0];
  // (undefined for a workgroup without a share: looked at only if w < P)
  const uint64_t info0 = (uint64_t)a.wg_info[2 * w + 2], info1 = (uint64_t)a.wg_info[2 * w + 3];
  auto store_dims = [&](int64_t r, const float (&x)[V]) __attribute__((always_inline)) {
    if (!head_ok) return;
    const int64_t at = r * a.io.out_stride_t + (int64_t)head * a.io.out_stride_h + sub * V;
#pragma unroll
    for (int i = 0; i < V; ++i) store_act_rt(a.io.out_dtype, a.io.out, at + i, x[i]);
  };
  // empty decode sequences (no tile: length 0): zeros, lse = -inf; the merging blocks share them out (the grid may hold one
  // more, the plan's)
  for (int s = w; s < B; s += a.num_wg) {
    const int q0e = a.cu_seqlens_q ? a.cu_seqlens_q[s] : s;
    const int q1e = a.cu_seqlens_q ? a.cu_seqlens_q[s + 1] : s + 1;
    if (q1e - q0e == 1 && a.seq_lens[s] <= 0) {
      float z[V];
#pragma unroll
      for (int i = 0; i < V; ++i) z[i] = 0.f;
      store_dims(q0e, z);
      if (a.io.lse != nullptr && sub == 0 && head_ok) a.io.lse[(int64_t)q0e * Hq + head] = -INFINITY;
    }
  }
  const int P = active_workgroups(total, a.num_wg);
  if (w == 0 || w >= P) return;
  const int seq = (int)(uint32_t)info0, w_first = (int)(uint32_t)info1, w_last = (int)(info1 >> 32);
  const int64_t row = (int64_t)(info0 >> 32);
  if (w_first == w_last) return;  // not cut
  const int span = w_last - w_first + 1;
  if (span > 16) {
    // A long span (one sequence over dozens of workgroups): a whole wave per q head, 64 slots per pass, and the
    // block's 16 heads spread over the first four blocks that begin inside the sequence (there are span - 1).
    constexpr int V2 = D / 64;
    const int j = w - (w_first + 1);
    const int h1 = (blockIdx.y * 4 + j) * 4 + (threadIdx.x >> 6);
    if (j < 0 || j >= 4 || h1 >= Hq) return;   // j < 0: the share begins with the sequence, not inside it
    float m = -INFINITY, l = 0.f, acc[V2];
#pragma unroll
    for (int i = 0; i < V2; ++i) acc[i] = 0.f;
    for (int wb = w_first; wb <= w_last; wb += kWave) {
      const int wj = wb + lane;
      const bool live = wj <= w_last;
      // loads are unconditional (clamped to the sequence's last workgroup) and what they return is removed with
      // a bit mask where the slot holds nothing
      const int64_t slot = (int64_t)min(wj, w_last) + seq;
      const uint32_t keep = live ? 0xffffffffu : 0u;
      const float mj_raw = a.part_ml[(slot * Hq + h1) * 2 + 0];
      const float lj_raw = a.part_ml[(slot * Hq + h1) * 2 + 1];
      const float mj = live ? as_f32(as_u32(mj_raw) & keep) : -INFINITY;
      const float lj = as_f32(as_u32(lj_raw) & keep);
      const float m_new = fmaxf(m, wave_max(mj));
      const float ca = __builtin_amdgcn_exp2f(m - m_new);  // first chunk: exp2(-inf) = 0
      const float ej = live ? __builtin_amdgcn_exp2f(mj - m_new) : 0.f;
      l = l * ca + wave_sum(lj * ej);
#pragma unroll
      for (int i = 0; i < V2; ++i) acc[i] *= ca;
      m = m_new;
      // up to sixty-four slots per round trip (128 registers of partial outputs in flight per lane)
      constexpr int kBatch = V2 <= 2 ? 64 : 128 / V2;
      const int count = min(kWave, w_last - wb + 1);
      for (int k0 = 0; k0 < count; k0 += kBatch) {
        float pv[kBatch][V2];
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
          const int64_t sk = (int64_t)min(wb + k0 + k, w_last) + seq;
          const float* po = a.part_o + (sk * Hq + h1) * (int64_t)D + lane * V2;
#pragma unroll
          for (int i = 0; i < V2; ++i) pv[k][i] = po[i];
        }
#pragma unroll
        for (int k = 0; k < kBatch; ++k) {
          const float wk = (k0 + k) < count ? lane_value(ej, (k0 + k) & (kWave - 1)) : 0.f;  // unnormalised sums
          const uint32_t kk = wk != 0.f ? 0xffffffffu : 0u;
#pragma unroll
          for (int i = 0; i < V2; ++i) acc[i] += as_f32(as_u32(pv[k][i]) & kk) * wk;
        }
      }
    }
    l += sink_term(a.io.sinks, h1, m);
    const float inv = 1.0f / l;
#pragma unroll
    for (int i = 0; i < V2; ++i)
      store_act_rt(a.io.out_dtype, a.io.out, row * a.io.out_stride_t + (int64_t)h1 * a.io.out_stride_h + lane * V2 + i, acc[i] * inv);
    if (a.io.lse != nullptr && lane == 0) a.io.lse[row * Hq + h1] = (m + __builtin_amdgcn_logf(l)) * kLn2;
    return;
  }
  if (w != w_first + 1) return;  // another block's to merge

  const float* po_head = a.part_o + (int64_t)head * D + sub * V;
  const float* ml_head = a.part_ml + (int64_t)head * 2;
  // lane `sub` of a group takes slot wb + sub's (m, l); the group agrees on the maximum and the weights, then
  // every lane adds up its dims over the slots.  All loads of a pass are unconditional (slots past the last
  // reread the last one and get weight 0; a select on a loaded value would become a branch around the load) and
  // leave before the first is used.  N slots per pass.
  float m = -INFINITY, l = 0.f, acc[V];
#pragma unroll
  for (int i = 0; i < V; ++i) acc[i] = 0.f;
  auto pass = [&](int wb, auto n_tag) __attribute__((always_inline)) {
    constexpr int N = decltype(n_tag)::value;   // <= 16
    const int wj = wb + sub;
    const bool live = sub < N && wj <= w_last;
    const int64_t slot = (int64_t)min(wj, w_last) + seq;
    const float mj_raw = ml_head[slot * Hq * 2 + 0];
    const float lj_raw = ml_head[slot * Hq * 2 + 1];
    float po[N][V];
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const int64_t sk = (int64_t)min(wb + k, w_last) + seq;
      const float* p = po_head + sk * Hq * (int64_t)D;
#pragma unroll
      for (int i = 0; i < V; i += 4) {
        const floatx4 x = *reinterpret_cast<const floatx4*>(p + i);
        po[k][i] = x.x; po[k][i + 1] = x.y; po[k][i + 2] = x.z; po[k][i + 3] = x.w;
      }
    }
    const uint32_t keep = live ? 0xffffffffu : 0u;
    const float mj = live ? as_f32(as_u32(mj_raw) & keep) : -INFINITY;
    const float lj = as_f32(as_u32(lj_raw) & keep);
    const float m_new = fmaxf(m, group_max<16>(mj));
    const float ca = __builtin_amdgcn_exp2f(m - m_new);  // first pass: exp2(-inf) = 0
    const float ej = live ? __builtin_amdgcn_exp2f(mj - m_new) : 0.f;
    l = l * ca + row16_sum(lj * ej);
    m = m_new;
#pragma unroll
    for (int i = 0; i < V; ++i) acc[i] *= ca;
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const float wk = __shfl(ej, grp + k, kWave);  // 0 for slots past the last and for empty ones
      const uint32_t kk = wk != 0.f ? 0xffffffffu : 0u;
#pragma unroll
      for (int i = 0; i < V; ++i) acc[i] += as_f32(as_u32(po[k][i]) & kk) * wk;
    }
  };
  constexpr int kLong = V <= 8 ? 16 : 8;   // 128 registers of partial outputs in flight per lane
  if (span <= 4) {
    pass(w_first, std::integral_constant<int, 4>{});
  } else if (span <= 8) {
    pass(w_first, std::integral_constant<int, 8>{});
  } else {
    for (int wb = w_first; wb <= w_last; wb += kLong) pass(wb, std::integral_constant<int, kLong>{});
  }
  l += sink_term(a.io.sinks, head, m);
  const float inv = 1.0f / l;
#pragma unroll
  for (int i = 0; i < V; ++i) acc[i] *= inv;
  store_dims(row, acc);
  if (a.io.lse != nullptr && sub == 0 && head_ok)
    a.io.lse[row * Hq + head] = (m + __builtin_amdgcn_logf(l)) * kLn2;
}

// The same merge with a grid over the sequences, for batches of few sequences (every one of which is cut, most
// of them several times): grid (num_seqs, ceil(Hq / 4)), 4 waves, one wave per q head, lane owns D/64 dims.  The
// sequence's place on the work line comes from the main kernel (seq_first_unit).
template <int D, bool PLAN>
__global__ __launch_bounds__(256) void paged_decode_streamk_reduce_by_seq_kernel(StreamKArgs a) {
  if constexpr (PLAN)
    if (plan_block(a)) return;
  constexpr int V = D / 64;
  const int lane = threadIdx.x & 63;
  const int head = blockIdx.y * 4 + (threadIdx.x >> 6);
  const int seq = blockIdx.x;
  if (head >= a.io.num_q_heads) return;
  // all the loads that depend on nothing but the arguments go out together, before the first branch
  const int q0 = a.cu_seqlens_q ? a.cu_seqlens_q[seq] : seq;
  const int q1 = a.cu_seqlens_q ? a.cu_seqlens_q[seq + 1] : seq + 1;
  const int len = a.seq_lens[seq];
  const int64_t total = a.wg_info[0];
  const int64_t start = a.seq_first_unit[seq];   // defined for every decode sequence that has a tile
  if (q1 - q0 != 1) return;
  const int64_t row = q0;
  const int ntiles = len > 0 ? decode_tiles(len, a.io.window) : 0;
  if (ntiles == 0) {  // empty sequence: defined output (zeros, lse = -inf)
    for (int i = 0; i < V; ++i)
      store_act_rt(a.io.out_dtype, a.io.out, row * a.io.out_stride_t + (int64_t)head * a.io.out_stride_h + lane * V + i, 0.f);
    if (a.io.lse != nullptr && lane == 0) a.io.lse[row * a.io.num_q_heads + head] = -INFINITY;
    return;
  }
  const int P = active_workgroups(total, a.num_wg);
  // the sequence's tiles are units start + setup_units .. start + setup_units + ntiles - 1
  const int w_first = wg_of_unit(start + a.setup_units, total, P);
  const int w_last = wg_of_unit(start + a.setup_units + ntiles - 1, total, P);
  if (w_first == w_last) return;  // written directly by the main kernel

  // pass 1: every lane takes one workgroup's (m, l); the wave agrees on the max and the weights
  // pass 2: weighted sum of the partial outputs, all loads independent of each other
  float m = -INFINITY, l = 0.f, acc[V];
#pragma unroll
  for (int i = 0; i < V; ++i) acc[i] = 0.f;
  // Few slots (the usual case: a sequence spans a handful of workgroups): the (m, l) pairs and ALL
  // the partial outputs are requested in one go, so the kernel pays one memory round trip for them
  // instead of two.
  constexpr int kFew = 32;
  // N = how many slots the one-round-trip path requests (all of them unconditionally: slots past the
  // last reread the last one), in three sizes so that a short span does not fetch 32 rows
  auto merge_few = [&](auto n_tag) __attribute__((always_inline)) {
    constexpr int N = decltype(n_tag)::value;
    const int w = w_first + lane;
    const bool live = w <= w_last;
    const int64_t slot = (int64_t)min(w, w_last) + seq;
    const uint32_t keep = live ? 0xffffffffu : 0u;
    const float mj_raw = a.part_ml[(slot * a.io.num_q_heads + head) * 2 + 0];
    const float lj_raw = a.part_ml[(slot * a.io.num_q_heads + head) * 2 + 1];
    float po[N][V];
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const int64_t sk = (int64_t)min(w_first + k, w_last) + seq;
      const float* p = a.part_o + (sk * a.io.num_q_heads + head) * (int64_t)D + lane * V;
#pragma unroll
      for (int i = 0; i < V; ++i) po[k][i] = p[i];
    }
    const float mj = live ? as_f32(as_u32(mj_raw) & keep) : -INFINITY;
    const float lj = as_f32(as_u32(lj_raw) & keep);
    m = wave_max(mj);
    const float ej = live ? __builtin_amdgcn_exp2f(mj - m) : 0.f;
    l = wave_sum(lj * ej);
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const float wk = lane_value(ej, k);  // 0 for slots past the last and for empty ones
      const uint32_t kk = wk != 0.f ? 0xffffffffu : 0u;
#pragma unroll
      for (int i = 0; i < V; ++i) acc[i] += as_f32(as_u32(po[k][i]) & kk) * wk;
    }
  };
  const int span = w_last - w_first + 1;
  if (span <= 4) {
    merge_few(std::integral_constant<int, 4>{});
  } else if (span <= 12) {
    merge_few(std::integral_constant<int, 12>{});
  } else if (span <= kFew) {
    merge_few(std::integral_constant<int, kFew>{});
  } else
  for (int wb = w_first; wb <= w_last; wb += kWave) {
    const int w = wb + lane;
    const bool live = w <= w_last;
    // loads are unconditional (clamped to the sequence's last workgroup) and what they return is
    // removed with a bit mask where the slot holds nothing: a select on the loaded value becomes a
    // branch around the load, and the loads of successive slots would then run one after another
    const int64_t slot = (int64_t)min(w, w_last) + seq;
    const uint32_t keep = live ? 0xffffffffu : 0u;
    const float mj_raw = a.part_ml[(slot * a.io.num_q_heads + head) * 2 + 0];
    const float lj_raw = a.part_ml[(slot * a.io.num_q_heads + head) * 2 + 1];
    const float mj = live ? as_f32(as_u32(mj_raw) & keep) : -INFINITY;
    const float lj = as_f32(as_u32(lj_raw) & keep);
    const float m_new = fmaxf(m, wave_max(mj));
    const float ca = __builtin_amdgcn_exp2f(m - m_new);  // first chunk: exp2(-inf) = 0
    const float ej = live ? __builtin_amdgcn_exp2f(mj - m_new) : 0.f;
    l = l * ca + wave_sum(lj * ej);
#pragma unroll
    for (int i = 0; i < V; ++i) acc[i] *= ca;
    m = m_new;
    // up to sixty-four slots per round trip (128 registers of partial outputs in flight per lane): a long span is
    // merged by ONE wave per (sequence, q head), so this path is a chain of round trips (a 256-slot span -- one
    // 128k-token sequence -- takes 21 us; 22.5 us with 16 slots per trip).  The loads of a batch are unconditional
    // (slots past the last reread the last one, weight 0) so that they all leave before the first is used.
    constexpr int kBatch = V <= 2 ? 64 : 128 / V;
    const int count = min(kWave, w_last - wb + 1);
    for (int k0 = 0; k0 < count; k0 += kBatch) {
      float pv[kBatch][V];
#pragma unroll
      for (int k = 0; k < kBatch; ++k) {
        const int64_t sk = (int64_t)min(wb + k0 + k, w_last) + seq;
        const float* po = a.part_o + (sk * a.io.num_q_heads + head) * (int64_t)D + lane * V;
#pragma unroll
        for (int i = 0; i < V; ++i) pv[k][i] = po[i];
      }
#pragma unroll
      for (int k = 0; k < kBatch; ++k) {
        const float wk = (k0 + k) < count ? lane_value(ej, (k0 + k) & (kWave - 1)) : 0.f;  // unnormalised sums
        const uint32_t kk = wk != 0.f ? 0xffffffffu : 0u;
#pragma unroll
        for (int i = 0; i < V; ++i) acc[i] += as_f32(as_u32(pv[k][i]) & kk) * wk;
      }
    }
  }
  l += sink_term(a.io.sinks, head, m);
  const float inv = 1.0f / l;
#pragma unroll
  for (int i = 0; i < V; ++i)
    store_act_rt(a.io.out_dtype, a.io.out, row * a.io.out_stride_t + (int64_t)head * a.io.out_stride_h + lane * V + i, acc[i] * inv);
  if (a.io.lse != nullptr && lane == 0)
    a.io.lse[row * a.io.num_q_heads + head] = (m + __builtin_amdgcn_logf(l)) * kLn2;
}

// The same merge for a handful of sequences, each cut dozens or hundreds of times (long contexts): grid
// (num_seqs, Hq), the block's four waves share ONE q head's span -- wave p takes the span's slots p, p + 4, ... --
// and their four states meet in LDS.  (With a wave per head a 256-slot span was a chain of eight round trips:
// 20.8 us for one 128k-token sequence, next to a 48 us main kernel.)
template <int D, bool PLAN>
__global__ __launch_bounds__(256) void paged_decode_streamk_reduce_split4_kernel(StreamKArgs a) {
  if constexpr (PLAN)
    if (plan_block(a)) return;
  constexpr int V = D / 64;
  __shared__ float sh_acc[3][V][kWave];
  __shared__ float sh_ml[3][2];
  const int lane = threadIdx.x & 63;
  const int part = threadIdx.x >> 6;
  const int head = blockIdx.y;
  const int seq = blockIdx.x;
  const int Hq = a.io.num_q_heads;
  const int q0 = a.cu_seqlens_q ? a.cu_seqlens_q[seq] : seq;
  const int q1 = a.cu_seqlens_q ? a.cu_seqlens_q[seq + 1] : seq + 1;
  const int len = a.seq_lens[seq];
  const int64_t total = a.wg_info[0];
  const int64_t start = a.seq_first_unit[seq];   // defined for every decode sequence that has a tile
  if (q1 - q0 != 1) return;                      // every branch down to the barrier is uniform over the block
  const int64_t row = q0;
  const int ntiles = len > 0 ? decode_tiles(len, a.io.window) : 0;
  if (ntiles == 0) {  // empty sequence: defined output (zeros, lse = -inf)
    if (part == 0) {
      for (int i = 0; i < V; ++i)
        store_act_rt(a.io.out_dtype, a.io.out, row * a.io.out_stride_t + (int64_t)head * a.io.out_stride_h + lane * V + i, 0.f);
      if (a.io.lse != nullptr && lane == 0) a.io.lse[row * Hq + head] = -INFINITY;
    }
    return;
  }
  const int P = active_workgroups(total, a.num_wg);
  const int w_first = wg_of_unit(start + a.setup_units, total, P);
  const int w_last = wg_of_unit(start + a.setup_units + ntiles - 1, total, P);
  if (w_first == w_last) return;  // written directly by the main kernel
  // this wave's slots: w_first + part + 4 i, i = 0 .. n - 1 (n = 0 for a span shorter than its number)
  const int span = w_last - w_first + 1;
  const int n = span > part ? (span - part + 3) / 4 : 0;
  float m = -INFINITY, l = 0.f, acc[V];
#pragma unroll
  for (int i = 0; i < V; ++i) acc[i] = 0.f;
  // one pass = N of the wave's slots from index i0 on: lane j takes slot j's (m, l), the wave agrees on the
  // maximum and the weights, every lane adds up its dims.  All loads are unconditional (indices past the last
  // reread the span's last slot and get weight 0) and leave before the first is used.
  auto pass = [&](int i0, auto n_tag) __attribute__((always_inline)) {
    constexpr int N = decltype(n_tag)::value;   // <= 64
    const int i = i0 + lane;
    const int wj = w_first + part + 4 * i;
    const bool live = lane < N && i < n;
    const int64_t slot = (int64_t)min(wj, w_last) + seq;
    const float mj_raw = a.part_ml[(slot * Hq + head) * 2 + 0];
    const float lj_raw = a.part_ml[(slot * Hq + head) * 2 + 1];
    float po[N][V];
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const int64_t sk = (int64_t)min(w_first + part + 4 * (i0 + k), w_last) + seq;
      const float* p = a.part_o + (sk * Hq + head) * (int64_t)D + lane * V;
#pragma unroll
      for (int x = 0; x < V; ++x) po[k][x] = p[x];
    }
    const uint32_t keep = live ? 0xffffffffu : 0u;
    const float mj = live ? as_f32(as_u32(mj_raw) & keep) : -INFINITY;
    const float lj = as_f32(as_u32(lj_raw) & keep);
    const float m_new = fmaxf(m, wave_max(mj));
    const float ca = m_new == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - m_new);   // a wave without a slot stays empty
    const float ej = live ? __builtin_amdgcn_exp2f(mj - m_new) : 0.f;
    l = l * ca + wave_sum(lj * ej);
    m = m_new;
#pragma unroll
    for (int x = 0; x < V; ++x) acc[x] *= ca;
#pragma unroll
    for (int k = 0; k < N; ++k) {
      const float wk = lane_value(ej, k);
      const uint32_t kk = wk != 0.f ? 0xffffffffu : 0u;
#pragma unroll
      for (int x = 0; x < V; ++x) acc[x] += as_f32(as_u32(po[k][x]) & kk) * wk;
    }
  };
  constexpr int kLong = V <= 2 ? 64 : 128 / V;   // 128 registers of partial outputs in flight per lane
  if (n <= 4) {
    pass(0, std::integral_constant<int, 4>{});
  } else if (n <= 16) {
    pass(0, std::integral_constant<int, 16>{});
  } else {
    for (int i0 = 0; i0 < n; i0 += kLong) pass(i0, std::integral_constant<int, kLong>{});
  }
  if (part > 0) {
#pragma unroll
    for (int x = 0; x < V; ++x) sh_acc[part - 1][x][lane] = acc[x];
    if (lane == 0) {
      sh_ml[part - 1][0] = m;
      sh_ml[part - 1][1] = l;
    }
  }
  __syncthreads();
  if (part > 0) return;
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    const float mp = sh_ml[p][0], lp = sh_ml[p][1];
    if (mp == -INFINITY) continue;   // that wave had no slot (uniform)
    const float m_new = fmaxf(m, mp);   // wave 0 always holds the span's first slot: m is finite
    const float ca = __builtin_amdgcn_exp2f(m - m_new), cb = __builtin_amdgcn_exp2f(mp - m_new);
    l = l * ca + lp * cb;
    m = m_new;
#pragma unroll
    for (int x = 0; x < V; ++x) acc[x] = acc[x] * ca + sh_acc[p][x][lane] * cb;
  }
  l += sink_term(a.io.sinks, head, m);
  const float inv = 1.0f / l;
#pragma unroll
  for (int x = 0; x < V; ++x)
    store_act_rt(a.io.out_dtype, a.io.out, row * a.io.out_stride_t + (int64_t)head * a.io.out_stride_h + lane * V + x, acc[x] * inv);
  if (a.io.lse != nullptr && lane == 0) a.io.lse[row * Hq + head] = (m + __builtin_amdgcn_logf(l)) * kLn2;
}

// ---- fixed partitions: grid (max_parts, num_seqs, head groups) --------------------------
struct V2Args {
  AttnIO io;
  const int32_t* seq_lens;
  float* tmp_out;
  float* max_logits;
  float* exp_sums;
  int partition_tiles;  // partition_size / 32
  int max_parts;
};

// BIAS: the instantiation with the ALiBi bias (DecodeTile's form with the extras; the soft cap stays the identity).
template <int D, int QDT, int WPW, bool BIAS>
__global__ __launch_bounds__(WPW * 64) void paged_decode_v2_kernel(V2Args a) {
  using DTile = DecodeTile<D, QDT, KVQ_F32>;
  __shared__ __align__(16) uint8_t lds[WPW][DTile::LDS_WAVE];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int hkv = __builtin_amdgcn_readfirstlane(blockIdx.z * WPW + wave);
  if (hkv >= a.io.g.num_kv_heads) return;
  const int part = blockIdx.x, seq = blockIdx.y;
  const int len = a.seq_lens[seq];
  const int ntiles = len > 0 ? (len + kTile - 1) / kTile : 0;
  const int t_begin = part * a.partition_tiles;
  if (t_begin >= ntiles) return;
  const int t_end = min(ntiles, t_begin + a.partition_tiles);
  typename DTile::State st;
  DTile::template run<BIAS>(a.io, DTile::lane_offsets(a.io.g, lane), seq, seq, len, 0, t_begin, t_end, hkv, lane, lds[wave], st);
  DTile::emit_v2(a.io, a.tmp_out, a.max_logits, a.exp_sums, seq, part, a.max_parts, hkv, lane, st);
}

// Main kernel + reduce of the balanced (or batch-invariant) split-K decode.
template <int D, int QDT>
int launch_streamk(const StreamKArgs& args, hipStream_t s) {
  const int hkv = args.io.g.num_kv_heads;
  int hpw = heads_per_wg(hkv);
  StreamKArgs a = args;
  // A handful of sequences: fewer kv heads per workgroup cut each of them into fewer, longer shares -- the waves of a head
  // meet in LDS instead of in the reduce's slots.  From 48 cuts per sequence on (5 sequences, 256 compute units); at
  // 24 the gain is gone (10 sequences of 1k - 8k: 31.1 us both ways, 2 of 20k with the fewest heads 27.8 for 26.9 us).
  // A step on MI355X, 8 kv heads of 128, before / after: 1 sequence of 2000 tokens 16.9 / 15.8 us, 16k 22.1 / 21.1,
  // 100k 49.5 / 47.0; 4 of 1k - 8k 24.5 / 22.6; 3 on 4 kv heads 21.0 / 18.5; token-major cache, 4 of 1k - 8k: 26.2 / 22.9.
  // Not at head size 256 (2 of 1k - 8k: 31.5 / 33.6), whose states are twice as long to fold.
  // One round of workgroups: more than eight kv heads would otherwise make two and more of them, of shares too short to be
  // worth it.
  if constexpr (D <= 128) {
    const int units = a.num_wg;
    while (!a.fixed_spans && hpw > 1 && a.num_wg > 48 * a.num_seqs) {
      hpw /= 2;
      a.num_wg /= 2;
    }
    const int groups = (hkv + hpw - 1) / hpw;
    if (hpw < heads_per_wg(hkv) && a.num_wg * groups > units) a.num_wg = units / groups > 1 ? units / groups : 1;
  }
  // a head's records of a block back to back (HND order): the tile loads may stream past the caches
  const bool stream = a.io.g.stride_slot == 2 * (code_bytes(a.io.g) + 4) && a.io.g.block_size >= 16;
  const bool extras = a.io.cap_c != 0.f || a.io.alibi != nullptr;   // the instantiation with soft cap and ALiBi
  if (a.whole) {
    const dim3 wgrid(hkv, a.num_seqs);
#define KVQ_WHOLE_FORM(C, CODE)                                                                                     \
  do {                                                                                                              \
    if (stream) hipLaunchKernelGGL((paged_decode_whole_kernel<D, QDT, C, CODE, true>), wgrid, dim3(512), 0, s, a);  \
    else hipLaunchKernelGGL((paged_decode_whole_kernel<D, QDT, C, CODE, false>), wgrid, dim3(512), 0, s, a);        \
  } while (0)
#define KVQ_WHOLE(CODE)                      \
  do {                                       \
    if (extras) KVQ_WHOLE_FORM(true, CODE);  \
    else KVQ_WHOLE_FORM(false, CODE);        \
  } while (0)
    if (a.io.g.code_type == KVQ_CODE_FP8_E4M3) KVQ_WHOLE(KVQ_CODE_FP8_E4M3);
    else if (a.io.g.code_type == KVQ_CODE_INT4) KVQ_WHOLE(KVQ_CODE_INT4);
    else KVQ_WHOLE(KVQ_CODE_INT8);
#undef KVQ_WHOLE
#undef KVQ_WHOLE_FORM
    return check_hip(hipGetLastError(), "paged_attn_int8 decode launch");
  }
  a.setup_units = setup_units_for(8 / hpw);
  dim3 grid(a.num_wg, (hkv + hpw - 1) / hpw);
#define KVQ_SK_FORM(H, C, CODE, S)                                                                                \
  do {                                                                                                            \
    if (a.fixed_spans)                                                                                            \
      hipLaunchKernelGGL((paged_decode_streamk_kernel<D, QDT, H, C, CODE, S, true>), grid, dim3(512), 0, s, a);   \
    else                                                                                                          \
      hipLaunchKernelGGL((paged_decode_streamk_kernel<D, QDT, H, C, CODE, S>), grid, dim3(512), 0, s, a);         \
  } while (0)
#define KVQ_SK_CODE(H, C, CODE)                                                                                   \
  do {                                                                                                            \
    if (stream) KVQ_SK_FORM(H, C, CODE, true);                                                                    \
    else KVQ_SK_FORM(H, C, CODE, false);                                                                          \
  } while (0)
#define KVQ_SK(H, C)                                                                                              \
  do {                                                                                                            \
    if (a.io.g.code_type == KVQ_CODE_FP8_E4M3) KVQ_SK_CODE(H, C, KVQ_CODE_FP8_E4M3);                              \
    else if (a.io.g.code_type == KVQ_CODE_INT4) KVQ_SK_CODE(H, C, KVQ_CODE_INT4);                                 \
    else KVQ_SK_CODE(H, C, KVQ_CODE_INT8);                                                                        \
  } while (0)
  if (extras) {
    switch (hpw) {
      case 8: KVQ_SK(8, true); break;
      case 4: KVQ_SK(4, true); break;
      case 2: KVQ_SK(2, true); break;
      default: KVQ_SK(1, true); break;
    }
  } else {
    switch (hpw) {
      case 8: KVQ_SK(8, false); break;
      case 4: KVQ_SK(4, false); break;
      case 2: KVQ_SK(2, false); break;
      default: KVQ_SK(1, false); break;
    }
  }
#undef KVQ_SK
#undef KVQ_SK_CODE
#undef KVQ_SK_FORM
  int rc = check_hip(hipGetLastError(), "paged_attn_int8 decode launch");
  if (rc) return rc;
  if (a.fixed_spans) {
    dim3 rgrid(a.num_seqs, (a.io.num_q_heads + 3) / 4);
    hipLaunchKernelGGL((paged_decode_fixed_spans_reduce_kernel<D>), rgrid, dim3(256), 0, s, a);
    return check_hip(hipGetLastError(), "paged_attn_int8 reduce launch");
  }
  // a sequence is cut where a share begins inside it: a batch of few sequences has most of them cut several
  // times (grid over the sequences, a wave per q head), a large batch has at most one cut per share and many
  // sequences with none (grid over the shares, four q heads per wave)
#define KVQ_REDUCE(K)                                                                      \
  do {                                                                                     \
    if (plan_blocks > 0) hipLaunchKernelGGL((K<D, true>), rgrid, dim3(256), 0, s, a);      \
    else hipLaunchKernelGGL((K<D, false>), rgrid, dim3(256), 0, s, a);                     \
  } while (0)
  const int plan_blocks = a.plan != nullptr ? 1 : 0;
  if (16 * a.num_seqs <= a.num_wg) {   // a handful of sequences, each cut many times: four waves per q head
    dim3 rgrid(a.num_seqs + plan_blocks, a.io.num_q_heads);
    KVQ_REDUCE(paged_decode_streamk_reduce_split4_kernel);
  } else if (8 * a.num_seqs <= 3 * a.num_wg) {
    dim3 rgrid(a.num_seqs + plan_blocks, (a.io.num_q_heads + 3) / 4);
    KVQ_REDUCE(paged_decode_streamk_reduce_by_seq_kernel);
  } else {
    dim3 rgrid(a.num_wg + plan_blocks, (a.io.num_q_heads + 15) / 16);
    KVQ_REDUCE(paged_decode_streamk_reduce_kernel);
  }
#undef KVQ_REDUCE
  return check_hip(hipGetLastError(), "paged_attn_int8 reduce launch");
}

template <int D, int QDT>
int launch_v2(const V2Args& a, int num_seqs, hipStream_t s) {
  const int hkv = a.io.g.num_kv_heads;
  const int wpw = heads_per_wg(hkv);
  dim3 grid(a.max_parts, num_seqs, (hkv + wpw - 1) / wpw);
#define KVQ_V2(W, BIAS) hipLaunchKernelGGL((paged_decode_v2_kernel<D, QDT, W, BIAS>), grid, dim3(W * 64), 0, s, a)
  if (a.io.alibi != nullptr) {
    switch (wpw) {
      case 8: KVQ_V2(8, true); break;
      case 4: KVQ_V2(4, true); break;
      case 2: KVQ_V2(2, true); break;
      default: KVQ_V2(1, true); break;
    }
  } else {
    switch (wpw) {
      case 8: KVQ_V2(8, false); break;
      case 4: KVQ_V2(4, false); break;
      case 2: KVQ_V2(2, false); break;
      default: KVQ_V2(1, false); break;
    }
  }
#undef KVQ_V2
  return check_hip(hipGetLastError(), "paged_attn_v2_int8 launch");
}

}  // namespace kvq
