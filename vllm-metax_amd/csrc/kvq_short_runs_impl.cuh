// Short query runs on a head-major cache (gfx950): 1 .. 64 columns (query token, q head of a kv group) per sequence, as a
// speculative-decoding step has them.
//
// The decode kernel's work split for runs of more than one token: the 32-token tiles of all items -- an item is up to
// 16 NT columns of one sequence -- form one line that is cut into equal shares, a workgroup of eight waves per compute
// unit takes a share, 8 / HPW waves of which share a kv head's tiles (HPW = 1, 2 or 4 kv heads).  Head sizes 64 and 128.  A run of
// tiles that covers its item writes the rows, any other leaves partial states for the reduce kernel.  One-token
// sequences of the batch are items like any other, so the launch needs neither the decode kernels nor the plan.
// With a workgroup per (sequence, kv head), whatever the sequence's length, a batch was as slow as its longest one:
// 24 sequences of 1k-8k tokens with 2-6 query tokens each took 97 us in that kernel, 2.4 TB/s; the step they are part
// of went from 105.8 to 71.3 us (now 70.1).
#pragma once

#include "kvq_prefill_tile.cuh"
#include "kvq_short_runs.h"
#include "kvq_work_line.cuh"

namespace kvq {

int heads_per_wg(int num_kv_heads);

struct ShortItem {
  int seq, q_begin, q_len, len, q0;
  int t0, t1;   // its tiles: those that hold a token some column sees (none: t0 == t1)
};
__device__ __forceinline__ int clamp_limit(int lim, int len) { return lim < 0 ? 0 : (lim > len ? len : lim); }
__device__ __forceinline__ ShortItem short_item(const ShortRunArgs& a, int item) {
  ShortItem it;
  it.seq = item / a.blocks;
  it.q0 = (item - it.seq * a.blocks) * a.q_tokens;
  it.q_begin = a.cu_seqlens_q[it.seq];
  it.q_len = a.cu_seqlens_q[it.seq + 1] - it.q_begin;
  it.len = max(a.seq_lens[it.seq], 0);
  const int ctx = it.len - it.q_len;
  const int last = clamp_limit(a.causal ? ctx + min(it.q0 + a.q_tokens, it.q_len) : it.len, it.len);
  const int first = a.io.window > 0 ? max(0, clamp_limit(ctx + it.q0 + 1, it.len) - a.io.window) : 0;
  it.t1 = it.q0 < it.q_len ? (last + kTile - 1) / kTile : 0;
  it.t0 = min(first / kTile, it.t1);
  return it;
}
__device__ __forceinline__ int short_units(const ShortItem& it, int setup) { return it.t1 > it.t0 ? it.t1 - it.t0 + setup : 0; }

// At most N of the wave's vector memory operations still under way (they complete in order).
template <int N>
__device__ __forceinline__ void wait_loads() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// LDS bytes of a wave: two windows, in which a state must fit when several waves serve one head.
template <int D, int CODE>
constexpr int short_runs_lds_wave() {
  using DTile = DecodeTile<D, KVQ_BF16, kRuntimeDtype, CODE, true>;
  return 2 * (DTile::LDS_TILE + 64 * 4) > DTile::LDS_STATE ? 2 * (DTile::LDS_TILE + 64 * 4) : DTile::LDS_STATE;
}

// EXT: soft cap and ALiBi (the plain kernel carries neither; the sliding window is in both).
template <int D, int NT, int HPW, int CODE, bool EXT>
__global__ __launch_bounds__(512) void short_runs_streamk_kernel(ShortRunArgs a) {
  using PT = PrefillTile<D, KVQ_BF16, kRuntimeDtype, NT, CODE, true>;   // (the query's type is read at run time)
  using DTile = typename PT::DTile;
  constexpr int NSUB = 8 / HPW;
  // two windows per wave: a tile streams into one, past the registers, while the other is computed (with a tile in
  // flight in registers the two column tiles' accumulators spilled: 420 against 106 us on the batch named above)
  constexpr int kWindow = DTile::LDS_TILE + 64 * 4;
  constexpr int kLdsWave = short_runs_lds_wave<D, CODE>();
  // (139 KB at head size 128, one workgroup per compute unit.  A fixed array: dynamic LDS of that size needs a function
  // attribute that the first call of each instantiation would set, possibly inside a stream capture.)
  __shared__ __align__(16) uint8_t lds_all[8 * kLdsWave];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sub = wave % NSUB;
  const int hkv = blockIdx.y * HPW + wave / NSUB;
  const AttnIO& io = a.io;
  if (hkv >= io.g.num_kv_heads) return;  // a finished wave no longer counts at the workgroup's barriers
  uint8_t* lds = lds_all + wave * kLdsWave;
  const int w = blockIdx.x;
  const int items = a.num_seqs * a.blocks;

  // the share [lo, hi) of the line, and the item that holds its first unit (each wave redoes the scan; up to 64 items are
  // held from the first pass, without the second trip for their lengths: 12 sequences on an int4 cache 32.4 -> 31.8 us)
  int64_t total = 0;
  int n0 = 0, incl0 = 0;   // the last 64 items' units and their running sum: of up to 64 items, all there is to know
  for (int base = 0; base < items; base += kWave) {
    const int i = base + lane;
    const int n = short_units(short_item(a, min(i, items - 1)), a.setup_units);
    n0 = i < items ? n : 0;
    incl0 = wave_incl_scan(n0);
    total += __builtin_amdgcn_readlane(incl0, 63);
  }
  const int num_wg = active_workgroups(total, a.num_wg);
  if (w == 0 && blockIdx.y == 0 && wave == 0 && lane == 0) a.line[0] = total;
  if (w >= num_wg) return;
  const int64_t lo = wg_tile_begin(w, total, num_wg), hi = wg_tile_begin(w + 1, total, num_wg);
  if (lo >= hi) return;
  int item = 0;
  int64_t start = 0;   // the item's first unit
  if (items <= kWave) {
    const int src = __builtin_ctzll(__builtin_amdgcn_ballot_w64(n0 > 0 && incl0 - n0 <= lo && lo < incl0));   // lo < total: there is one
    item = src;
    start = __builtin_amdgcn_readlane(incl0 - n0, src);
  } else {
    int64_t cum = 0;
    for (int base = 0; base < items; base += kWave) {
      const int i = base + lane;
      const int n = i < items ? short_units(short_item(a, min(i, items - 1)), a.setup_units) : 0;
      const int incl = wave_incl_scan(n);
      const uint64_t hit = __builtin_amdgcn_ballot_w64(n > 0 && cum + incl - n <= lo && lo < cum + incl);
      if (hit != 0) {
        const int src = __builtin_ctzll(hit);
        item = base + src;
        start = cum + __builtin_amdgcn_readlane(incl - n, src);
        break;
      }
      cum += __builtin_amdgcn_readlane(incl, 63);
    }
  }

  const LaneOffsets off = DTile::lane_offsets(io.g, lane);
  const float sc_mul = lane < 32 ? io.scale_log2 * DTile::kKScaleMul : kPScale;
  const uint32_t wspan = io.window > 0 ? (uint32_t)io.window : 0x7fffffffu;
  const int c = lane & 15;

  int64_t pos = lo;
  for (; pos < hi && item < items; ++item) {
    const ShortItem it = short_item(a, item);
    const int units = short_units(it, a.setup_units);
    if (units == 0) continue;
    const int u_begin = (int)(pos - start);
    const int u_end = hi - start < units ? (int)(hi - start) : units;
    const int tb = it.t0 + (u_begin > a.setup_units ? u_begin - a.setup_units : 0);
    const int te = it.t0 + u_end - a.setup_units;
    const int64_t item_start = start;
    pos = start + u_end;
    start += units;
    if (tb >= te) continue;   // this share ends inside the setup charge and holds no tile

    // ---- the first tile leaves, then the columns and their query rows
    const int32_t* bt_row = io.block_table + (int64_t)it.seq * io.bt_stride;
    int t = tb + sub;
    const bool has_tiles = t < te;   // (a wave without a tile loads one all the same and uses nothing)
    TileBlocks nb = DTile::fetch_blocks(io, bt_row, it.len, t);
    uint8_t *cur = lds, *next = lds + kWindow;
    DTile::load_tile_to_lds(DTile::window(io, nb, t, hkv), off, lane, cur);
    DTile::phase_fence();
    nb = DTile::fetch_blocks(io, bt_row, it.len, t + NSUB);
    const int ctx = it.len - it.q_len;
    // column nt * 16 + c: query token (nt * 16 + c) / group of the item (recomputed where it is needed: the registers of
    // the tile loop are scarce)
    auto column = [&](int nt, int64_t& row, int& head, int& qi) __attribute__((always_inline)) {
      const int n = nt * 16 + c;
      const int qt = n / io.group;
      qi = it.q0 + qt;
      const bool ok = qt < a.q_tokens && qi < it.q_len;
      head = hkv * io.group + (ok ? n - qt * io.group : 0);
      row = it.q_begin + (ok ? qi : it.q0);
      return ok;
    };
    int limit[NT];
    float s_init[NT], ali[NT];
    half8_t qb[NT][PT::KSTEPS];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      int64_t row;
      int head, qi;
      const bool valid = column(nt, row, head, qi);
      limit[nt] = valid ? clamp_limit(a.causal ? ctx + qi + 1 : it.len, it.len) : 0;
      ali[nt] = EXT ? alibi_slope(io.alibi, head) : 0.f;
      const int64_t elem = row * io.q_stride_t + (int64_t)head * io.q_stride_h;
      if (a.q_dtype == KVQ_BF16)
        s_init[nt] = DTile::load_q_row(io, elem, valid, lane, qb[nt]);
      else if (a.q_dtype == KVQ_F16)
        s_init[nt] = DecodeTile<D, KVQ_F16, kRuntimeDtype, CODE, true>::load_q_row(io, elem, valid, lane, qb[nt]);
      else
        s_init[nt] = DecodeTile<D, KVQ_F32, kRuntimeDtype, CODE, true>::load_q_row(io, elem, valid, lane, qb[nt]);
    }
    // tiles every column sees whole need no mask
    const int min_limit = clamp_limit(a.causal ? ctx + it.q0 + 1 : it.len, it.len);
    const int max_limit = clamp_limit(a.causal ? ctx + min(it.q0 + a.q_tokens, it.q_len) : it.len, it.len);
    const int max_first = io.window > 0 ? max(0, max_limit - io.window) : 0;

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
    auto softmax = [&]() __attribute__((always_inline)) {
      if ((t + 1) * kTile <= min_limit && t * kTile >= max_first)
        PT::template qk_softmax<false, EXT>(io, off, qb, s_init, limit, wspan, t, lane, cur, st, p_op, ali);
      else
        PT::template qk_softmax<true, EXT>(io, off, qb, s_init, limit, wspan, t, lane, cur, st, p_op, ali);
    };
    if (has_tiles) {
      while (t + NSUB < te) {
        // the other window was read to the end: it takes the next tile
        DTile::load_tile_to_lds(DTile::window(io, nb, t + NSUB, hkv), off, lane, next);
        nb = DTile::fetch_blocks(io, bt_row, it.len, t + 2 * NSUB);
        wait_loads<DTile::kDmaLoads>();   // all but those just issued: tile t is there
        DTile::stage_scales(off, sc_mul, lane, cur);
        softmax();
        PT::pv_any(t * kTile < max_first, off, p_op, cur, st);   // not the sequence's last tile
        DTile::phase_fence();
        uint8_t* done = cur;
        cur = next;
        next = done;
        t += NSUB;
      }
      wait_loads<0>();
      DTile::stage_scales(off, sc_mul, lane, cur);
      softmax();
      PT::template pv<true>(off, p_op, cur, st);
    } else {
      wait_loads<0>();   // nothing is under way to the window when the wave goes on
    }
    if (tb == it.t0 && blockIdx.y == 0 && wave == 0 && lane == 0) a.line[1 + item] = item_start;   // for the reduce kernel
    if constexpr (NSUB > 1) {
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        if (nt > 0) lds_barrier();   // the windows take the next column tile's states
        if (sub != 0 && has_tiles) PT::dump_state(st, nt, lane, lds);
        lds_barrier();
        if (sub == 0) {
#pragma unroll
          for (int j = 1; j < NSUB; ++j)
            if (tb + j < te) PT::fold_state(st, nt, lane, lds + j * kLdsWave);   // wave j owned a tile
        }
      }
      lds_barrier();   // the windows may be overwritten by the next run
    }
    if (sub == 0) {
      const bool whole = tb == it.t0 && te == it.t1;
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        int64_t row;
        int head, qi;
        const bool valid = column(nt, row, head, qi);
        if (whole) {
          PT::emit(io, nt, row, head, valid, lane, st);
          continue;
        }
        const float l = PT::total_l(st, nt);
        if (!valid) continue;
        const int slot = 2 * w + (tb == it.t0 ? 1 : 0);
        const int64_t at = (uint32_t)((slot * io.g.num_kv_heads + hkv) * a.rows + nt * 16 + c);
        float v[D / 4];
        PT::gather_row(st, nt, 1.0f / DTile::kOutDiv, v);
        const int g = lane >> 4;
#pragma unroll
        for (int i = 0; i < D / 4; i += 4)
          *reinterpret_cast<floatx4*>(a.part_o + at * D + DTile::out_dim(g, i)) = (floatx4){v[i], v[i + 1], v[i + 2], v[i + 3]};
        if (g == 0) {
          a.part_ml[2 * at] = st.m[nt];
          a.part_ml[2 * at + 1] = l;
        }
      }
    }
  }
}

// Merges the partial states of the items that more than one workgroup touched, and gives the rows of items without a
// tile their defined output (zeros, lse = -inf).  grid (items, ceil(q_tokens Hq / 4)), a wave per (query token, q head),
// a lane owns D / 64 dims; lane j of a pass takes slot j's (m, l), every load of a pass leaves before the first is used
// (slots past the last reread it and weigh 0; a select on a loaded value would become a branch around the load).
template <int D>
__global__ __launch_bounds__(256) void short_runs_reduce_kernel(ShortRunArgs a) {
  constexpr int V = D / 64;
  const int lane = threadIdx.x & 63;
  const int r = blockIdx.y * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const AttnIO& io = a.io;
  const int Hq = io.num_q_heads;
  const int qt = r / Hq, head = r - qt * Hq;
  const int item = blockIdx.x;
  const int64_t total = a.line[0], start = a.line[1 + item];   // (start: defined for an item with tiles)
  const ShortItem it = short_item(a, item);
  if (qt >= a.q_tokens || it.q0 + qt >= it.q_len) return;
  const int64_t row = it.q_begin + it.q0 + qt;
  const int64_t out_at = row * io.out_stride_t + (int64_t)head * io.out_stride_h + lane * V;
  float acc[V];
#pragma unroll
  for (int i = 0; i < V; ++i) acc[i] = 0.f;
  float m = -INFINITY, l = 0.f;
  const int ntiles = it.t1 - it.t0;
  if (ntiles > 0) {
    const int P = active_workgroups(total, a.num_wg);
    const int w_first = wg_of_unit(start + a.setup_units, total, P);
    const int w_last = wg_of_unit(start + a.setup_units + ntiles - 1, total, P);
    if (w_first == w_last) return;  // written by the main kernel
    const int hkv = head / io.group, n = qt * io.group + head - hkv * io.group;
    const int64_t stride = (int64_t)io.g.num_kv_heads * a.rows;   // rows between two slots
    const int64_t at0 = (int64_t)hkv * a.rows + n;
    // workgroup w's state of this item lies at at0 + 2 w stride, the first one's (it begins with the item) a stride further
    auto pass = [&](int wb, auto n_tag) __attribute__((always_inline)) {
      constexpr int N = decltype(n_tag)::value;
      const int wj = wb + lane;
      const bool live = lane < N && wj <= w_last;
      const int64_t mine = at0 + (2 * (int64_t)min(wj, w_last) + (wj == w_first ? 1 : 0)) * stride;
      const float mj_raw = a.part_ml[2 * mine], lj_raw = a.part_ml[2 * mine + 1];
      float po[N][V];
#pragma unroll
      for (int k = 0; k < N; ++k) {
        const int64_t at = at0 + 2 * (int64_t)min(wb + k, w_last) * stride + (k == 0 && wb == w_first ? stride : 0);
        const float* p = a.part_o + at * D + lane * V;
#pragma unroll
        for (int i = 0; i < V; ++i) po[k][i] = p[i];
      }
      const uint32_t keep = live ? 0xffffffffu : 0u;
      const float mj = live ? as_f32(as_u32(mj_raw) & keep) : -INFINITY;
      const float lj = as_f32(as_u32(lj_raw) & keep);
      const float m_new = fmaxf(m, wave_max(mj));
      const float m_ref = m_new == -INFINITY ? 0.f : m_new;   // a column may have seen nothing yet
      const float ca = __builtin_amdgcn_exp2f(m - m_ref);
      const float ej = live ? __builtin_amdgcn_exp2f(mj - m_ref) : 0.f;
      l = l * ca + wave_sum(lj * ej);
      m = m_new;
#pragma unroll
      for (int i = 0; i < V; ++i) acc[i] *= ca;
#pragma unroll
      for (int k = 0; k < N; ++k) {
        const float wk = lane_value(ej, k);
        const uint32_t kk = wk != 0.f ? 0xffffffffu : 0u;
#pragma unroll
        for (int i = 0; i < V; ++i) acc[i] += as_f32(as_u32(po[k][i]) & kk) * wk;
      }
    };
    if (w_last - w_first < 4) pass(w_first, std::integral_constant<int, 4>{});
    else
      for (int wb = w_first; wb <= w_last; wb += 16) pass(wb, std::integral_constant<int, 16>{});
    if (l > 0.f) l += sink_term(io.sinks, head, m);   // a row without a visible key keeps its zeros
  }
  const float inv = l > 0.f ? 1.0f / l : 0.f;
#pragma unroll
  for (int i = 0; i < V; ++i) store_act_rt(io.out_dtype, io.out, out_at + i, acc[i] * inv);
  if (io.lse != nullptr && lane == 0) io.lse[row * Hq + head] = l > 0.f ? (m + __builtin_amdgcn_logf(l)) * kLn2 : -INFINITY;
}

template <int D, int NT, int HPW, int CODE, bool EXT>
static int launch_one(const ShortRunArgs& a, dim3 grid, hipStream_t s) {
  hipLaunchKernelGGL((short_runs_streamk_kernel<D, NT, HPW, CODE, EXT>), grid, dim3(512), 0, s, a);
  return check_hip(hipGetLastError(), "paged_attn_int8 short runs launch");
}

// Instantiated once per head size in kvq_short_runs_d<head size>.hip.
template <int D>
int launch_short_runs_d(const ShortRunArgs& args, hipStream_t s) {
  ShortRunArgs a = args;
  const int hkv = a.io.g.num_kv_heads;
  // Kv heads per workgroup: fewer of them cut the line into fewer, longer shares (the waves of a head meet in LDS), so
  // that an item leaves fewer partial states -- a state is up to 32 columns of D floats per head, and with a cut per 8 heads
  // a batch wrote and read 27 MB of them beside 173 MB of cache.  Four rather than eight (MI355X, a step, 8 kv heads of 128,
  // 2 - 6 query tokens on 1k - 8k): 24 sequences 73.5 -> 71.1 us, 40: 83.4 -> 79.8, 64: 125.2 -> 119.7; 90 short ones
  // 55.0 -> 54.7.  Head size 64, 24 sequences 43.7 -> 41.2; int4 codes 54.9 -> 53.7, 64: 102.8 -> 102.3; 2 kv heads, 64 sequences
  // 76.7 -> 77.8, with int4 codes 66.3 -> 66.5, fewer of them gain.  Below four a share's start weighs more than the states saved (24 sequences, 4 kv heads: 2 per
  // workgroup 50.6 for 47.9 us) until an item is cut dozens of times: one sequence of 16k tokens 34.5 -> 24.9 us, 5 of
  // 8k - 16k on 16 kv heads 62.8 -> 60.3; 12 on 4 kv heads (21 cuts each) would lose, 38.9 -> 41.1.
  int hpw = heads_per_wg(hkv);
  while (hpw > 4 || (hpw > 1 && a.num_wg > 24 * a.num_seqs * a.blocks)) {
    hpw /= 2;
    a.num_wg /= 2;
  }
  // One round of workgroups: with more than eight kv heads there would be two and more of them.  A step, captured, with a
  // workgroup per eight heads / without this bound / with it: 32 kv heads, a run of 3 tokens on 4000 27.5 / 42.2 / 20.4 us, 8 on
  // 1500 43.1 / 47.8 / 27.8; 16 kv heads, 4 on 1500 21.8 / 24.9 / 18.3, 24 on 1k - 8k 105.1 / 100.7 / 87.8.
  const int groups = (hkv + hpw - 1) / hpw;
  if (hpw < heads_per_wg(hkv) && a.num_wg * groups > args.num_wg) a.num_wg = args.num_wg / groups > 1 ? args.num_wg / groups : 1;
  a.setup_units = setup_units_for(8 / hpw);
  dim3 grid(a.num_wg, (hkv + hpw - 1) / hpw);
  const bool ext = a.io.cap_c != 0.f || a.io.alibi != nullptr;
#define KVQ_SR_CODE(NT, H, CODE)                                                              \
  do {                                                                                                                     \
    if (ext) rc = launch_one<D, NT, H, CODE, true>(a, grid, s);                                                            \
    else rc = launch_one<D, NT, H, CODE, false>(a, grid, s);                                                               \
  } while (0)
#define KVQ_SR(NT, H)                                                                  \
  do {                                                                                 \
    if (a.io.g.code_type == KVQ_CODE_FP8_E4M3) KVQ_SR_CODE(NT, H, KVQ_CODE_FP8_E4M3);  \
    else if (a.io.g.code_type == KVQ_CODE_INT4) KVQ_SR_CODE(NT, H, KVQ_CODE_INT4);     \
    else KVQ_SR_CODE(NT, H, KVQ_CODE_INT8);                                            \
  } while (0)
#define KVQ_SR_HPW(NT)          \
  do {                          \
    switch (hpw) {              \
      case 4: KVQ_SR(NT, 4); break; \
      case 2: KVQ_SR(NT, 2); break; \
      default: KVQ_SR(NT, 1); break; \
    }                           \
  } while (0)
  int rc = KVQ_OK;
  if (a.cols == 32) KVQ_SR_HPW(2);
  else KVQ_SR_HPW(1);
#undef KVQ_SR_HPW
#undef KVQ_SR
#undef KVQ_SR_CODE
  if (rc) return rc;
  dim3 rgrid(a.num_seqs * a.blocks, (a.q_tokens * a.io.num_q_heads + 3) / 4);
  hipLaunchKernelGGL((short_runs_reduce_kernel<D>), rgrid, dim3(256), 0, s, a);
  return check_hip(hipGetLastError(), "paged_attn_int8 short runs reduce launch");
}

}  // namespace kvq
