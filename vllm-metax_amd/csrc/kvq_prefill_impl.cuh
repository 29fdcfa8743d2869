// Chunked-prefill tile over the int8 paged cache (gfx950, wave64, MFMA f16): query runs longer
// than one token, causal, reading context and the run's own tokens from the cache.
//
// The MFMA N dimension carries (query token, q head of the group) pairs -- the
// folding of query tokens and the q heads of a kv group that the unified attention op the reference
// calls does (vllm_metax/v1/attention/backends/triton_attn.py:43, 688-725) -- so one pass over a kv head's
// records serves 16 * NT columns: the records are read from HBM, dropped into the wave's LDS
// window and turned into fp16 operands once per tile, and each operand feeds NT MFMAs.
// One wavefront = one (sequence, query block, kv head); it streams tiles 0 .. last visible tile
// with the decode tile's load / stage machinery and applies the causal limit per column.
#pragma once

#include <type_traits>

#include "kvq_prefill_tile.cuh"

namespace kvq {

constexpr int kMaxKSplit = 8;   // context splits of a launch at most
constexpr int kRunsInKernel = 16;   // sequences of a launch up to which the shared tile needs no plan (find_run)

struct PrefillArgs {
  AttnIO io;
  const int32_t* seq_lens;
  const int32_t* cu_seqlens_q;
  int num_seqs;
  int causal;
  int q_tokens;  // query tokens per block: (16 * NT) / group
  // [1 + B]: how many sequences of the batch have a query run (q_len > 1, len > 0), then their numbers; written
  // ahead of the attention kernel of the same call (write_prefill_plan); nullptr where the workgroup-shared tile
  // finds the runs itself (find_run).
  const int32_t* plan;
  // Context splits of the workgroup-shared tile (1 = none).  With S > 1 an item's tiles are cut into S ranges, each
  // range is a workgroup of its own that leaves a partial state per (query row, q head) in `part`
  // ([row][q head][split][D + 2] fp32: the accumulated row, the reference maximum, the sum), and a merge kernel
  // combines them: a launch with few items on a long context (a small prefill chunk of one long request) would
  // otherwise walk the whole context in a handful of workgroups, one tile after the other.
  int ksplit;
  int num_tokens;   // rows of q, with ksplit > 1
  float* part;
  // Batch-invariant mode: which runs a kernel of this launch takes -- 0 all, 1 only those that fill the
  // workgroup-shared tile by themselves (q_len x group >= 64), 2 only the others.  Without the mode the batch's
  // longest run chooses ONE kernel for every run of the launch, so a short run's bits would depend on its company.
  int route;
};

// grid (query blocks of the longest run, sequences, ceil(Hkv / WPW)); wave w of a workgroup owns
// kv head (head group) * WPW + w.  Sequences with a one-token run belong to the decode kernel.
// SPLIT: grid z = Hkv and ALL waves of the workgroup serve one kv head, taking the
// item's tiles in turn (wave w: tiles t_start + w, + WPW, ...); their states are folded in LDS at the end.  For
// launches with few items and long contexts -- a handful of query tokens per sequence, as a speculative-decoding
// step has them: one wave per item leaves most of the chip's waves idle (measured on MI355X, 64 sequences of
// 1k-8k tokens with 2 or 4 query tokens each: 280 us per call that way against 118 us for one query token).
template <int D, int QDT, int ODT, int NT, int WPW, int CODE = KVQ_CODE_INT8, bool SPLIT = false>
__global__ __launch_bounds__(WPW * 64) void paged_prefill_kernel(PrefillArgs a) {
  using PT = PrefillTile<D, QDT, ODT, NT, CODE, false, D == 256 && WPW == 8>;
  using DTile = typename PT::DTile;
  __shared__ __align__(16) uint8_t lds_all[WPW][DTile::LDS_WAVE];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // which sequence, head group and query block: the linear workgroup number read over the plan's sequences,
  // sequence by sequence (longest first), inside a sequence query-block-major over the head groups, longest
  // block first, the head group shifted by the block number (see paged_prefill_shared_kernel)
  const unsigned nqb = gridDim.x, hz = gridDim.z, per_seq = nqb * hz;
  const unsigned lin = blockIdx.x + nqb * (blockIdx.y + gridDim.y * blockIdx.z);
  if (lin >= per_seq * (unsigned)a.plan[0]) return;   // uniform over the workgroup
  const unsigned rem = lin % per_seq, qbi = rem / hz;
  const int seq = a.plan[1 + lin / per_seq];
  const int hkv = SPLIT ? (int)((rem % hz + qbi) % hz) : (int)((rem % hz + qbi) % hz) * WPW + wave;
  constexpr int STEP = SPLIT ? WPW : 1;          // tiles between two of this wave's
  const AttnIO& io = a.io;
  if (hkv >= io.g.num_kv_heads) return;
  const int q_begin = a.cu_seqlens_q[seq];
  const int q_len = a.cu_seqlens_q[seq + 1] - q_begin;
  const int len = a.seq_lens[seq];
  const int q0 = (int)(nqb - 1 - qbi) * a.q_tokens;   // first query token of this block within the run
  if (q_len <= 1 || q0 >= q_len || len <= 0) return;
  if (a.route == 2 && q_len * io.group >= 64) return;   // the workgroup-shared tile's (uniform over the workgroup)
  uint8_t* lds = lds_all[wave];

  // ---- columns: n = nt * 16 + c  ->  (query token q0 + n / group, head n % group)
  const int c = lane & 15;
  const int ctx = len - q_len;                      // tokens before the run
  int limit[NT];                                    // visible tokens of the lane's column
  int64_t row[NT];
  int head[NT];
  bool valid[NT];
  int max_limit = 0, min_limit = 0x7fffffff;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int n = nt * 16 + c;
    const int qt = n / io.group;
    const int qi = q0 + qt;
    valid[nt] = qt < a.q_tokens && qi < q_len;
    head[nt] = hkv * io.group + (n - qt * io.group);
    row[nt] = q_begin + (valid[nt] ? qi : q0);
    int lim = a.causal ? ctx + qi + 1 : len;
    lim = lim < 0 ? 0 : (lim > len ? len : lim);
    limit[nt] = valid[nt] ? lim : 0;
    max_limit = max(max_limit, limit[nt]);
    min_limit = min(min_limit, valid[nt] ? lim : 0x7fffffff);
  }
  max_limit = wave_max_i32(max_limit);
  min_limit = -wave_max_i32(-min_limit);
  const int t_end = (max_limit + kTile - 1) / kTile;  // wave-uniform
  // sliding window: a column sees [limit - window, limit); the wave starts at the tile that holds
  // the earliest of these lower edges and masks tiles below the latest one
  const uint32_t wspan = io.window > 0 ? (uint32_t)io.window : 0x7fffffffu;
  const int min_first = io.window > 0 ? max(0, min(min_limit, max_limit) - io.window) : 0;
  const int max_first = io.window > 0 ? max(0, max_limit - io.window) : 0;
  const int t_start = min_first / kTile;
  if (t_end == 0) {  // nothing visible for any column (run longer than the sequence): defined zeros
    typename PT::State z;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
      for (int dt = 0; dt < PT::DT; ++dt) z.o[nt][dt] = (floatx4){0.f, 0.f, 0.f, 0.f};
      z.psum[nt] = (floatx4){0.f, 0.f, 0.f, 0.f};
      z.m[nt] = -INFINITY;
      z.l[nt] = 0.f;
      if (!SPLIT || wave == 0) PT::emit(io, nt, row[nt], head[nt], valid[nt], lane, z);
    }
    return;
  }

  const LaneOffsets lo = DTile::lane_offsets(io.g, lane);
  const int32_t* bt_row = io.block_table + (int64_t)seq * io.bt_stride;
  typename DTile::Tile kv;
  int t = t_start + (SPLIT ? wave : 0);
  const bool has_tiles = t < t_end;              // without the split: always
  // (a wave without a tile still loads one -- the block table is read clamped into the sequence -- and uses nothing)
  TileBlocks nb = DTile::fetch_blocks(io, bt_row, len, t);
  DTile::load_tile(io, DTile::window(io, nb, t, hkv), lo, kv);
  DTile::phase_fence();
  nb = DTile::fetch_blocks(io, bt_row, len, t + STEP);

  half8_t qb[NT][PT::KSTEPS];
  float s_init[NT], ali[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) ali[nt] = alibi_slope(io.alibi, valid[nt] ? head[nt] : hkv * io.group);
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
    s_init[nt] = DTile::load_q_row(io, row[nt] * io.q_stride_t + (int64_t)(valid[nt] ? head[nt] : hkv * io.group) * io.q_stride_h,
                                   valid[nt], lane, qb[nt]);
  const float sc_mul = lane < 32 ? io.scale_log2 * DTile::kKScaleMul : kPScale;
  typename PT::State st;
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
#pragma unroll
    for (int dt = 0; dt < PT::DT; ++dt) st.o[nt][dt] = (floatx4){0.f, 0.f, 0.f, 0.f};
    st.psum[nt] = (floatx4){0.f, 0.f, 0.f, 0.f};
    st.m[nt] = -INFINITY;
    st.l[nt] = 0.f;
  }
  half8_t p_op[NT];
  if (has_tiles) {
    while (t + STEP < t_end) {
      const typename DTile::Window w = DTile::window(io, nb, t + STEP, hkv);
      DTile::stage(kv, lo, sc_mul, lane, lds);
      DTile::phase_fence();
      DTile::load_tile(io, w, lo, kv);
      DTile::phase_fence();
      nb = DTile::fetch_blocks(io, bt_row, len, t + 2 * STEP);
      if ((t + 1) * kTile <= min_limit && t * kTile >= max_first)
        PT::template qk_softmax<false>(io, lo, qb, s_init, limit, wspan, t, lane, lds, st, p_op, ali);
      else
        PT::template qk_softmax<true>(io, lo, qb, s_init, limit, wspan, t, lane, lds, st, p_op, ali);
      PT::pv_any(t * kTile < max_first, lo, p_op, lds, st);   // not the item's last tile
      DTile::phase_fence();
      t += STEP;
    }
    DTile::stage(kv, lo, sc_mul, lane, lds);
    PT::template qk_softmax<true>(io, lo, qb, s_init, limit, wspan, t, lane, lds, st, p_op, ali);
    PT::template pv<true>(lo, p_op, lds, st);
  }
  if constexpr (SPLIT) {
    // every wave of the workgroup arrives here (the returns above are uniform over it)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      if (nt > 0) lds_barrier();   // the windows are read no more: they take the next column tile's states
      if (wave != 0 && has_tiles) PT::dump_state(st, nt, lane, lds);
      lds_barrier();
      if (wave == 0) {
#pragma unroll
        for (int j = 1; j < WPW; ++j)
          if (t_start + j < t_end) PT::fold_state(st, nt, lane, lds_all[j]);   // wave j owned a tile
      }
    }
    if (wave != 0) return;
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) PT::emit(io, nt, row[nt], head[nt], valid[nt], lane, st);
}

// Launches with this many items (query block x sequence x kv head) or fewer spread each item over a workgroup's waves.
constexpr int64_t kSplitItems = 2048;

template <int D, int QDT, int ODT, int NT, int WPW, int CODE = KVQ_CODE_INT8>
static int launch_prefill_cfg(const PrefillArgs& a, int max_query_len, hipStream_t s) {
  const int blocks = (max_query_len + a.q_tokens - 1) / a.q_tokens;
  if (blocks > 0x7fffffff / 2 || a.num_seqs > 65535) return fail(KVQ_EINVAL, "paged_attn_int8: prefill grid out of range");
  // (not in the batch-invariant mode: how an item is cut would depend on what else the launch holds)
  if (!batch_invariant() && (int64_t)blocks * a.num_seqs * a.io.g.num_kv_heads <= kSplitItems &&
      a.io.g.num_kv_heads <= 65535) {
    // waves per item: eight with one column tile per wave; four with two, and for 8-bit codes of head size 256 (their
    // accumulators, and there a tile in flight beside them, need the registers of a 256-thread workgroup.  In eight waves of
    // head size 256 up to 42 words went to scratch and came back in every tile, each time behind a wait for the tile in
    // flight: 24 sequences of 1k-8k tokens with 2-6 query tokens, 16/8 heads, 527 us a step, 254 with the eight waves' steps
    // in order and 142 with four; one of 512 tokens on 16k 1852, 755, 471.  int4 tiles are half the registers: 295, 81, 103.)
    constexpr int SW = NT == 1 && (D < 256 || CODE == KVQ_CODE_INT4) ? 8 : 4;
    dim3 grid(blocks, a.num_seqs, a.io.g.num_kv_heads);
    hipLaunchKernelGGL((paged_prefill_kernel<D, QDT, ODT, NT, SW, CODE, true>), grid, dim3(SW * 64), 0, s, a);
    return check_hip(hipGetLastError(), "paged_prefill launch");
  }
  dim3 grid(blocks, a.num_seqs, (a.io.g.num_kv_heads + WPW - 1) / WPW);
  hipLaunchKernelGGL((paged_prefill_kernel<D, QDT, ODT, NT, WPW, CODE>), grid, dim3(WPW * 64), 0, s, a);
  return check_hip(hipGetLastError(), "paged_prefill launch");
}

// The workgroup-shared tile (kvq_prefill_shared.cuh), head sizes 64 and 128.
template <int D>
int launch_prefill_shared(PrefillArgs& a, int max_query_len, int q_dtype, int out_dtype, hipStream_t s);

// Runs that fill the workgroup-shared tile's columns take it.
inline bool takes_shared_tile(int head_size, int max_query_len, int group) { return head_size <= 128 && max_query_len * group >= 64; }

template <int D, int QDT, int ODT>
static int launch_prefill_nt(PrefillArgs& a, int max_query_len, hipStream_t s);

// Batch-invariant mode: every run goes to the kernel its OWN length chooses.  Runs that fill the workgroup-shared
// tile by themselves take it; the others take the per-wave tile with one column tile per wave -- in a second launch
// when the batch holds both kinds.
template <int D, int QDT, int ODT>
static int launch_prefill_invariant(PrefillArgs& a, int max_query_len, hipStream_t s) {
  const int group = a.io.group;
  if (takes_shared_tile(D, max_query_len, group)) {
    a.route = 1;
    if (int e = launch_prefill_nt<D, QDT, ODT>(a, max_query_len, s)) return e;
    a.route = 2;
    const int longest_short = (63 / group);        // q_len x group < 64
    if (longest_short < 2) return KVQ_OK;           // no run of two tokens or more is short
    return launch_prefill_nt<D, QDT, ODT>(a, longest_short, s);
  }
  a.route = 0;
  return launch_prefill_nt<D, QDT, ODT>(a, max_query_len, s);
}

template <int D, int QDT, int ODT>
static int launch_prefill_nt(PrefillArgs& a, int max_query_len, hipStream_t s) {
  constexpr int WPW = 4;
  const bool fp8 = a.io.g.code_type == KVQ_CODE_FP8_E4M3;
  const bool int4 = a.io.g.code_type == KVQ_CODE_INT4;
  // long runs: the workgroup-shared fp16 tile (compute-bound shape), for every kind of code
  if constexpr (D <= 128) {
    if (takes_shared_tile(D, max_query_len, a.io.group) && a.route != 2) return launch_prefill_shared<D>(a, max_query_len, QDT, ODT, s);
  }
  if (fp8) {  // short runs of fp8 codes: the per-wave tile, one column tile per wave
    a.q_tokens = 16 / a.io.group;
    return launch_prefill_cfg<D, QDT, ODT, 1, WPW, KVQ_CODE_FP8_E4M3>(a, max_query_len, s);
  }
  if (int4) {
    a.q_tokens = 16 / a.io.group;
    return launch_prefill_cfg<D, QDT, ODT, 1, WPW, KVQ_CODE_INT4>(a, max_query_len, s);
  }
  // two column tiles per wave where the accumulators fit the register file next to a tile in flight
  if (D <= 128 && a.io.group * 2 <= 32 && max_query_len * a.io.group > 16 && !batch_invariant()) {
    a.q_tokens = 32 / a.io.group;
    return launch_prefill_cfg<D, QDT, ODT, (D <= 128 ? 2 : 1), WPW>(a, max_query_len, s);
  }
  a.q_tokens = 16 / a.io.group;
  return launch_prefill_cfg<D, QDT, ODT, 1, WPW>(a, max_query_len, s);
}

template <int D, int QDT>
static int launch_prefill_o(PrefillArgs& a, int max_query_len, int out_dtype, hipStream_t s) {
  switch (out_dtype) {
    case KVQ_F32: return batch_invariant() ? launch_prefill_invariant<D, QDT, KVQ_F32>(a, max_query_len, s)
                                           : launch_prefill_nt<D, QDT, KVQ_F32>(a, max_query_len, s);
    case KVQ_BF16: return batch_invariant() ? launch_prefill_invariant<D, QDT, KVQ_BF16>(a, max_query_len, s)
                                            : launch_prefill_nt<D, QDT, KVQ_BF16>(a, max_query_len, s);
    case KVQ_F16: return batch_invariant() ? launch_prefill_invariant<D, QDT, KVQ_F16>(a, max_query_len, s)
                                           : launch_prefill_nt<D, QDT, KVQ_F16>(a, max_query_len, s);
    default: return fail(KVQ_EINVAL, "paged_attn_int8: unknown out_dtype %d", out_dtype);
  }
}

// Instantiated once per head size in kvq_prefill_d<head size>.hip.
template <int D>
int launch_prefill_q(PrefillArgs& a, int max_query_len, int q_dtype, int out_dtype, hipStream_t s) {
  switch (q_dtype) {
    case KVQ_F32: return launch_prefill_o<D, KVQ_F32>(a, max_query_len, out_dtype, s);
    case KVQ_BF16: return launch_prefill_o<D, KVQ_BF16>(a, max_query_len, out_dtype, s);
    case KVQ_F16: return launch_prefill_o<D, KVQ_F16>(a, max_query_len, out_dtype, s);
    default: return fail(KVQ_EINVAL, "paged_attn_int8: unknown q_dtype %d", q_dtype);
  }
}

}  // namespace kvq
