// Varlen attention with LSE output for the MLA prefill (gfx950): the step between the latent cache's
// gather + dequantise and the LSE merge of the chunked-context loop, and the causal pass over the new
// tokens.  K arrives as the two pieces the layer already has -- k_nope [S, H, NOPE] out of kv_b_proj and
// the rope part k_pe [S, ROPE] shared by all heads -- so the concatenated [S, H, NOPE + ROPE] tensor is
// never built.
//
// Workgroup = 128 query rows of one (sequence, head): 4 waves x 2 blocks of 16 rows.  The keys are walked 32
// at a time; a tile's K rows (NOPE + ROPE wide) and V rows stream from memory straight into LDS once per workgroup, one
// tile ahead, double-buffered (one barrier per tile), and every wave feeds its two row blocks from there, so a K or V byte
// is fetched from L2 once per 128 rows.  Which bytes a load's lanes bring is chosen so that the operand reads of K (chunks
// xor-swizzled by the row) and of V (successive rows from different loads, 32 bytes apart) meet no bank twice.
// What bounds it: latency -- matrix unit 44 % busy, vector unit 39 %, LDS 22 %.  Hence no registers between memory and LDS
// (they took 20 of them and a fifth of the tile's instructions), three workgroups per compute unit, and operands of either
// product requested four ahead of their use: K from the step's start, the first V while the softmax runs.  A step in which no product exceeds its row's maximum reduces nothing over lanes and rescales nothing.  Lane
// numbers, limits and the K addresses of a step are worked out anew for it: kept, they were 18 registers more than the 168
// there are at three workgroups.
// Measured: 4 requests with 300-1500 new tokens on 1000-2300 cached ones, 128 heads, a layer step 1335 -> 1192 us without the
// registers; then, side by side, with two operand reads under way, a wait for the next tile's loads in front of the V reads, a
// maximum reduced in every step and pairs of a causal launch one after the other / now: 1215 / 1176 (of which 484 us are the
// two kv_b_proj products); one request of 200 tokens on 4900 cached ones at 16 heads 215 / 200, three of 500-1500 at 64 heads
// 161 / 144, one of 1400 in fp16 at 32 heads 98 / 84.
// Both products are computed transposed so that every per-row quantity is lane-local:
//   S^T = K Q^T   A = K rows (lane = key, 8 consecutive d), B = Q (lane = query row): 16x16x32 MFMA of the
//                 input type; a lane ends up with 8 keys of ITS query row, so the row maximum is a
//                 reduction over the four quarter-waves and alpha / l stay in the lane.
//   O^T = V^T P^T B = P~ straight from the S^T registers (k slot j of quarter g is key 16 (j / 4) + 4 g +
//                 j % 4; any order works as long as V uses the same one).  A = V^T needs 8 keys of one
//                 dim per lane while a V row holds the dims of one key together: the LDS's transposing read
//                 (ds_read_b64_tr_b16) hands a lane four keys of one dim out of four rows, two of them make an
//                 operand, no register shuffles.  Output block i holds dims 16 i .. 16 i + 15; a lane ends
//                 with dims 16 i + 4 g .. + 3 of its own query row: 8-byte stores.
// Masked keys (beyond the sequence, or above the causal diagonal, which is aligned to the END of the
// keys as flash-attention does) get weight 0; their rows are clamped copies of the last valid key.
#include "kvq_attn_core.cuh"
#include "kvq_internal.h"

namespace kvq {

struct VarlenArgs {
  const void* q;
  const void* k_nope;
  const void* k_pe;
  const void* v;
  void* out;
  float* lse;
  const int32_t* cu_q;
  const int32_t* cu_k;
  int64_t q_st, q_sh, kn_st, kn_sh, kpe_st, v_st, v_sh, out_st, out_sh, total_q;
  int causal;
  int merge;   // out and lse hold the rows' state over other keys: this launch's is merged into it
  int last_pairs;   // (sequence, head) pairs of an XCD, the last ones, whose blocks are taken in turn (by_block_pairs)
  float scale_log2;
};

// acc + the two 16-bit floats of `pair` (fp16 or bf16).
template <int DT>
__device__ __forceinline__ float pair_sum(uint32_t pair, float acc) {
  if constexpr (DT == KVQ_F16) {
    const half2_t one = {(half_t)1.0f, (half_t)1.0f};
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, pair), one, acc, false);
  } else {
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    const bf16x2_t one = {(__bf16)1.0f, (__bf16)1.0f};
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, pair), one, acc, false);
  }
}

// The two 16-bit floats of `pair`.
template <int DT>
__device__ __forceinline__ void unpack2(uint32_t pair, float& lo, float& hi) {
  if constexpr (DT == KVQ_F16) {
    const half2_t h = __builtin_bit_cast(half2_t, pair);
    lo = (float)h.x;
    hi = (float)h.y;
  } else {
    lo = as_f32(pair << 16);
    hi = as_f32(pair & 0xffff0000u);
  }
}

// Where the pieces of a 32-key tile lie in LDS.  A tile goes from memory straight into LDS: a wave's load fills 1 KB there,
// lane i's 16 bytes at 16 i, and which bytes of the tensors a lane brings is free to choose.
template <int NOPE, int ROPE, int DV>
struct VarlenTile {
  // K, the nope and the rope part each: rows back to back, chunk ch of row r in slot ch ^ swizzle(r).  The 16 lanes that an
  // operand read (16 rows x the same chunk, 4 chunks per wave) serves at a time then meet every bank once.
  template <int W>
  __host__ __device__ static constexpr int swizzle(int r) { return W == 128 ? (r & 15) : W == 64 ? ((r >> 1) & 7) : ((r >> 2) & 3); }
  static constexpr int KN_BYTES = 32 * NOPE * 2, KR_BYTES = 32 * ROPE * 2;
  // V: a load brings 1 KB / row bytes rows that lie V_LOADS apart, and loads are 32 bytes apart, so that the four
  // successive rows of which a transposing read takes 32 bytes each lie on different banks.
  static constexpr int V_ROW = DV * 2, V_LOADS = 32 * V_ROW / 1024, V_PITCH = 1024 + 32;
  __host__ __device__ static constexpr int v_at(int r) { return (r % V_LOADS) * V_PITCH + (r / V_LOADS) * V_ROW; }
  static constexpr int V_AT = KN_BYTES + KR_BYTES, BYTES = V_AT + V_LOADS * V_PITCH;

  // Load j of a K part of width W: the lane's byte offset from the tile's first row.
  template <int W>
  __device__ static __forceinline__ uint32_t k_offset(int j, int lane, int64_t row_bytes) {
    constexpr int C = W / 8;
    const int r = j * (64 / C) + lane / C, ch = (lane % C) ^ swizzle<W>(r);
    return (uint32_t)(r * (int)row_bytes + 16 * ch);
  }
  __device__ static __forceinline__ uint32_t v_offset(int j, int lane, int64_t row_bytes) {
    constexpr int C = DV / 8;
    return (uint32_t)((j + V_LOADS * (lane / C)) * (int)row_bytes + 16 * (lane % C));
  }
  __device__ static __forceinline__ void load(__amdgpu_buffer_rsrc_t w, uint32_t offset, uint8_t* dst) {
    typedef __attribute__((address_space(3))) void* lds_ptr_t;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(w, (lds_ptr_t)dst, 16, offset, 0, 0, 0);
  }
};

template <int FROM, int TO, class F>
__device__ __forceinline__ void static_for(F f) {
  if constexpr (FROM < TO) {
    f(std::integral_constant<int, FROM>{});
    static_for<FROM + 1, TO>(f);
  }
}

// log2 of the XCDs that a launch's (sequence, head) pairs are dealt out to, every eighth pair to one of eight; 0: not at all.
__host__ __device__ constexpr unsigned xcd_bits_of(unsigned pairs) { return (pairs & 7u) == 0 ? 3 : 0; }

// Three waves per SIMD, i.e. workgroups per compute unit.  Two, of the same instructions, are no better where a launch has no
// more (launch alone, two / three per unit: 128 heads, 300 new tokens on 4000, 384 workgroups, 139.8 / 140.2 us, 500, 512,
// 168.0 / 169.7) and worse beyond (600, 640, 244.4 / 212.3; 64 heads, 1500 on 3000, 768, 194.0 / 173.8).
constexpr int kPerUnit = 3;

template <int DT, int NOPE, int ROPE, int DV>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kPerUnit, kPerUnit))) void varlen_attn_kernel(VarlenArgs a) {
  using VT = VarlenTile<NOPE, ROPE, DV>;
  constexpr int KSN = NOPE / 32, KSR = ROPE / 32, KS = KSN + KSR;   // k-steps of the QK product
  constexpr int DPL = DV / 16;                                      // dims per lane and output block
  constexpr int RB = 2;                                             // row blocks of 16 per wave
  // fp16 weights are kept 2^8 larger so that small ones stay normal; l carries the same factor
  constexpr float kShift = DT == KVQ_F16 ? 8.f : 0.f;
  constexpr int AHEAD = 4 < 2 * KS ? 4 : 2 * KS, AHEAD_V = 4 < DPL ? 4 : DPL;   // K and V operands requested ahead of their products
  __shared__ __align__(16) uint8_t lds[2][VT::BYTES];
  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Workgroups go to the eight XCDs in turn by their linear number, and every XCD has its own L2.  The query
  // blocks of one (sequence, head) all stream the same keys: numbered so that they land on ONE XCD (possible when
  // the (sequence, head) pairs divide by eight), its L2 serves all but the first reader of a tile.
  // Under the causal mask a pair's blocks differ in length, and one pair after the other, longest block first, the launch
  // ends on the long blocks of the last pairs: the last a.last_pairs of an XCD's pairs are taken block by block over all of
  // them (by_block_pairs says when and how many).
  int seq, head, qb;
  {
    const unsigned pairs = gridDim.y * gridDim.z, blocks = gridDim.x;
    const unsigned xcd_bits = xcd_bits_of(pairs);
    const unsigned lin = blockIdx.x + blocks * (blockIdx.y + gridDim.y * blockIdx.z);
    const unsigned j = lin >> xcd_bits, per_xcd = pairs >> xcd_bits;   // the XCD's j-th workgroup
    unsigned pair = j / blocks;
    qb = (int)(j - pair * blocks);
    const unsigned last = (unsigned)a.last_pairs;
    if (pair >= per_xcd - last) {
      const unsigned r = j - (per_xcd - last) * blocks;
      qb = (int)(r / last);
      pair = per_xcd - last + (r - (unsigned)qb * last);
    }
    pair = (pair << xcd_bits) + (lin & ((1u << xcd_bits) - 1));   // every eighth pair is this XCD's
    seq = (int)(pair / gridDim.y);
    head = (int)(pair - (unsigned)seq * gridDim.y);
  }
  const int q_begin = a.cu_q[seq], q_len = a.cu_q[seq + 1] - q_begin;
  const int k_begin = a.cu_k[seq], k_len = a.cu_k[seq + 1] - k_begin;
  // the last query blocks see the most keys under the causal mask: they are launched first
  const int q0wg = ((int)gridDim.x - 1 - qb) * (64 * RB);
  if (q0wg >= q_len) return;   // uniform over the workgroup
  const int c = lane & 15, g = lane >> 4;
  // key j is visible to query row i iff j <= i + (k_len - q_len)
  const int diag = k_len - q_len;
  const int wg_rows_end = min(q_len, q0wg + 64 * RB);
  const int wg_k_end = a.causal ? max(0, min(k_len, wg_rows_end - 1 + diag + 1)) : k_len;
  const int num_tiles = (wg_k_end + 31) / 32;
  if (a.merge && num_tiles == 0) return;   // nothing to add to the rows (uniform over the workgroup)

  // the lane number, worked out anew (kept from tile to tile it, and what follows from it, take registers)
  auto lane_anew = []() __attribute__((always_inline)) {
    uint32_t n;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(n));
    return (int)n;
  };
  // ---- the wave's rows
  int q0[RB], blk_k_end[RB], min_limit = k_len;
  auto limit_of = [&](int rb, int row) __attribute__((always_inline)) {   // keys that row `row` of a row block sees
    return a.causal ? max(0, min(k_len, q0[rb] + row + diag + 1)) : k_len;
  };
  u32x4 qop[RB][KS];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    q0[rb] = q0wg + (wave * RB + rb) * 16;
    const int qrow = min(q0[rb] + c, q_len - 1);   // rows past the end compute on a copy and are not stored
    const uint16_t* qp = static_cast<const uint16_t*>(a.q) + (int64_t)(q_begin + qrow) * a.q_st + (int64_t)head * a.q_sh + 8 * g;
#pragma unroll
    for (int s = 0; s < KS; ++s) qop[rb][s] = *reinterpret_cast<const u32x4*>(qp + 32 * s);
    min_limit = min(min_limit, limit_of(rb, 0));
    blk_k_end[rb] = q0[rb] >= q_len ? 0 : (a.causal ? max(0, min(k_len, q0[rb] + 15 + diag + 1)) : k_len);
  }
  const int wave_tiles = (max(blk_k_end[0], blk_k_end[1]) + 31) / 32;   // tiles this wave has anything to do in
  // the smallest limit among the wave's rows: tiles that end at or below it are visible to every row
  const int wave_min_limit = min_limit;

  floatx4 oacc[RB][DPL];
  float off[RB], top[RB], l[RB];   // kShift - row maximum; the largest product; lane's sum of weights
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
#pragma unroll
    for (int i = 0; i < DPL; ++i) oacc[rb][i] = (floatx4){0.f, 0.f, 0.f, 0.f};
    off[rb] = kShift;
    top[rb] = -INFINITY;
    l[rb] = 0.f;
  }

  // ---- tile loads.  "Buffer resource + a lane offset that never changes": the resources (scalar registers) are re-based on
  //      the tile's first key, a step per tile.  A resource ends with the tile's, hence also the sequence's, last key: rows
  //      past it read as zeros and are masked.  Every wave brings the same share of each part.
  constexpr int NL = VT::KN_BYTES / 4096, RL = VT::KR_BYTES / 1024, VL = VT::V_LOADS / 4;   // nope and V loads per wave; rope loads
  const uint8_t* kn_base = reinterpret_cast<const uint8_t*>(static_cast<const uint16_t*>(a.k_nope) + (int64_t)head * a.kn_sh);
  const uint8_t* kpe_base = reinterpret_cast<const uint8_t*>(a.k_pe);
  const uint8_t* v_base = reinterpret_cast<const uint8_t*>(static_cast<const uint16_t*>(a.v) + (int64_t)head * a.v_sh);
  const int64_t kn_row = a.kn_st * 2, kpe_row = a.kpe_st * 2, v_row_bytes = a.v_st * 2;   // bytes per key
  uint32_t n_off[NL], r_off = 0, v_off[VL];
#pragma unroll
  for (int i = 0; i < NL; ++i) n_off[i] = VT::template k_offset<NOPE>(wave * NL + i, lane, kn_row);
  const int rj = RL > 0 ? wave % (RL > 0 ? RL : 1) : 0;   // (fewer rope loads than waves: two waves bring the same)
  if constexpr (RL > 0) r_off = VT::template k_offset<ROPE>(rj, lane, kpe_row);
#pragma unroll
  for (int i = 0; i < VL; ++i) v_off[i] = VT::v_offset(wave * VL + i, lane, v_row_bytes);
  const uint8_t *kn_p = kn_base + (int64_t)k_begin * kn_row, *kpe_p = kpe_base + (int64_t)k_begin * kpe_row,
                *v_p = v_base + (int64_t)k_begin * v_row_bytes;   // the next tile's first key
  int left = k_len;                                               // keys from there on
  auto part = [&](const uint8_t*& p, int64_t row_bytes, int keys) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t w = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p), 0, keys * (int)row_bytes, 0x00020000);
    p += 32 * row_bytes;
    return w;
  };
  auto fetch = [&](uint8_t* buf) __attribute__((always_inline)) {
    const int keys = min(left, 32);
    left -= 32;
    const __amdgpu_buffer_rsrc_t rn = part(kn_p, kn_row, keys);
#pragma unroll
    for (int i = 0; i < NL; ++i) VT::load(rn, n_off[i], buf + (wave * NL + i) * 1024);
    if constexpr (RL > 0) VT::load(part(kpe_p, kpe_row, keys), r_off, buf + VT::KN_BYTES + rj * 1024);
    const __amdgpu_buffer_rsrc_t rv = part(v_p, v_row_bytes, keys);
#pragma unroll
    for (int i = 0; i < VL; ++i) VT::load(rv, v_off[i], buf + VT::V_AT + (wave * VL + i) * VT::V_PITCH);
  };
  // every load into LDS of this wave has landed, every LDS read is done, and so for the other waves
  auto tile_barrier = []() __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  // operand places of the lane: K row c, chunk g of a k-step (a k-step is four chunks); V rows 4 g + c / 4.  The chunk of
  // k-step s is that of the first one xor 4 s: worked out anew in every step, a register per part is all that is kept.
  uint32_t kn_read = (uint32_t)(c * NOPE * 2 + (g ^ VT::template swizzle<NOPE>(c)) * 16);
  uint32_t kr_read = ROPE > 0 ? (uint32_t)(VT::KN_BYTES + c * ROPE * 2 + (g ^ VT::template swizzle<ROPE>(c)) * 16) : 0;
  const uint32_t v_read = (uint32_t)(VT::V_AT + VT::v_at(4 * g + (c >> 2)) + 8 * (c & 3));

  // V^T operand of output block i, half h (keys 4 g .. + 3 and 16 + 4 g ..): the LDS's transposing read.  Lane s of a
  // quarter-wave names the 8 bytes [key kb + s / 4][dims 16 i + 4 (s % 4) .. + 3] and receives [keys kb .. kb + 3][dim 16 i + s].
  // In assembly because the compiler waits for every load under way, the next tile's too, in front of the builtin; so the
  // waits for what these read are written out as well.  To the compiler a read's registers hold their values at once:
  // tests/test_lds_read_waits.py follows the compiled code for a copy, a spill or a reuse before the wait.
  struct VOperand {
    u32x2 half[2];
  };
  auto read_v = [&](uint32_t at, auto block, VOperand& o) __attribute__((always_inline)) {
    constexpr int I = decltype(block)::value;
    asm volatile("ds_read_b64_tr_b16 %0, %2 offset:%3\n\tds_read_b64_tr_b16 %1, %2 offset:%4"
                 : "=&v"(o.half[0]), "=&v"(o.half[1]) : "v"(at), "n"(32 * I), "n"(VT::v_at(16) + 32 * I));
  };
  auto wait_v = [&](auto behind, VOperand& o) __attribute__((always_inline)) {   // `behind`: operands requested after this one
    asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(o.half[0]), "+v"(o.half[1]) : "n"(2 * decltype(behind)::value));
  };
  auto fence = []() __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); };

  auto step_fn = [&](int t, const uint8_t* buf) __attribute__((always_inline)) {
    // a wave at its products and softmax outranks the waves of its SIMD that wait at the barrier
    __builtin_amdgcn_s_setprio(1);
    // ---- S^T = K Q^T for the tile's two blocks of 16 keys, both row blocks off one operand read
    floatx4 sacc[RB][2];
    u32x4 ka[2 * KS];
    asm volatile("" : "+v"(kn_read), "+v"(kr_read));   // (what follows from them is not to be kept either)
    auto read_k = [&](int i) __attribute__((always_inline)) {
      const int blk = i / KS, s = i % KS;
      const uint8_t* p = s < KSN ? buf + (kn_read ^ (64 * s)) + blk * 16 * NOPE * 2 : buf + (kr_read ^ (64 * (s - KSN))) + blk * 16 * ROPE * 2;
      ka[i] = *reinterpret_cast<const u32x4*>(p);
    };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) read_k(i);
    fence();
#pragma unroll
    for (int i = 0; i < 2 * KS; ++i) {
#pragma unroll
      for (int rb = 0; rb < RB; ++rb)
        sacc[rb][i / KS] = mfma16<DT>(ka[i], qop[rb][i % KS], i % KS == 0 ? (floatx4){0.f, 0.f, 0.f, 0.f} : sacc[rb][i / KS]);
      if (i + AHEAD < 2 * KS) read_k(i + AHEAD);
      fence();
    }
    // the first V operands come in while the softmax runs
    VOperand va[DPL];
    const uint32_t v_at = v_read + (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint8_t*)buf;
    static_for<0, AHEAD_V>([&](auto i) __attribute__((always_inline)) { read_v(v_at, i, va[i]); });
    fence();
    // ---- online softmax in base 2, per row block
    // only a tile that reaches past some row's limit (the causal diagonal, the end of the keys) is masked: a uniform
    // branch round the compares and selects, which work on the products where they lie
    if ((t + 1) * 32 > wave_min_limit) {
      const int of = lane_anew();
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        const int visible = limit_of(rb, of & 15) - t * 32 - 4 * (of >> 4);
#pragma unroll
        for (int j = 0; j < 8; ++j)
          sacc[rb][j >> 2][j & 3] = 16 * (j >> 2) + (j & 3) < visible ? sacc[rb][j >> 2][j & 3] : -INFINITY;
      }
    }
    // A row's maximum moves where some lane's product exceeds it; in a step without such a lane neither the reduction over a
    // row's four lanes nor any rescaling is due.  It is the true maximum, whose weight is then exactly 1: a maximum that stays
    // put until exceeded by 2^8 saves more (four requests at 128 heads 1086 us, 1135 so) but has that weight rounded like any
    // other, and the error against float64 was 2 to 16 % larger.
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      // the maximum is taken over the raw products (the scale is positive and the same for every key), so that
      // scale and maximum enter each logit in ONE multiply-add
      float mx = -INFINITY;
#pragma unroll
      for (int j = 0; j < 8; ++j) mx = fmaxf(mx, sacc[rb][j >> 2][j & 3]);
      if (__builtin_amdgcn_ballot_w64(mx > top[rb]) != 0) {
        const float new_top = fmaxf(top[rb], max_over_quarters(mx));
        const float new_off = new_top == -INFINITY ? off[rb] : kShift - new_top * a.scale_log2;
        const float alpha = top[rb] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(new_off - off[rb]);
        top[rb] = new_top;
        off[rb] = new_off;
        l[rb] *= alpha;
#pragma unroll
        for (int i = 0; i < DPL; ++i) oacc[rb][i] *= alpha;
      }
    }
    u32x4 pk[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
      float p[8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        p[j] = __builtin_amdgcn_exp2f(__builtin_fmaf(sacc[rb][j >> 2][j & 3], a.scale_log2, off[rb]));   // a masked key: 2^-inf = 0
      pk[rb].x = pack2<DT>(p[0], p[1]);
      pk[rb].y = pack2<DT>(p[2], p[3]);
      pk[rb].z = pack2<DT>(p[4], p[5]);
      pk[rb].w = pack2<DT>(p[6], p[7]);
      // the row sum is that of the weights as the second product sees them (rounded to the input type): one
      // two-element dot product with ones per packed pair instead of two additions
#pragma unroll
      for (int w = 0; w < 4; ++w) l[rb] = pair_sum<DT>(pk[rb][w], l[rb]);
    }
    fence();
    // ---- O^T += V^T P^T
    static_for<0, DPL>([&](auto ic) __attribute__((always_inline)) {
      constexpr int I = decltype(ic)::value, BEHIND = I + AHEAD_V <= DPL ? AHEAD_V - 1 : DPL - 1 - I;
      wait_v(std::integral_constant<int, BEHIND>{}, va[I]);
      const u32x4 vt = {va[I].half[0].x, va[I].half[0].y, va[I].half[1].x, va[I].half[1].y};
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) oacc[rb][I] = mfma16<DT>(vt, pk[rb], oacc[rb][I]);
      if constexpr (I + AHEAD_V < DPL) read_v(v_at, std::integral_constant<int, I + AHEAD_V>{}, va[I + AHEAD_V]);
      fence();
    });
    __builtin_amdgcn_s_setprio(0);
  };
  if (num_tiles > 0) {
    fetch(lds[0]);
    tile_barrier();
  }
  for (int t = 0; t < num_tiles; t += 2) {
    if (t + 1 < num_tiles) fetch(lds[1]);
    if (t < wave_tiles) step_fn(t, lds[0]);
    tile_barrier();
    if (t + 1 < num_tiles) {
      if (t + 2 < num_tiles) fetch(lds[0]);
      if (t + 1 < wave_tiles) step_fn(t + 1, lds[1]);
      tile_barrier();
    }
  }

  const int lane_end = lane_anew(), c_end = lane_end & 15, g_end = lane_end >> 4;
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const float l_tot = sum_over_quarters(l[rb]);
    const bool live = l_tot > 0.f;
    float mul = live ? 1.f / l_tot : 0.f;
    if (q0[rb] + c_end >= q_len) continue;
    const int64_t tok = q_begin + q0[rb] + c_end;
    uint16_t* op = static_cast<uint16_t*>(a.out) + tok * a.out_st + (int64_t)head * a.out_sh;
    float lse = live ? __logf(l_tot) - off[rb] * kLn2 : -INFINITY;
    if (a.merge) {
      // The algebra of merge_attn_states, in the epilogue: the other keys' rows are read and the sum is written once.
      // (As a launch of its own the merge read both states and wrote the rows: 46 us of 1352 for 2765 rows x 128 heads.)
      float* const lp = a.lse + (int64_t)head * a.total_q + tok;
      const float given = *lp;
      const float prior = given == INFINITY ? -INFINITY : given;   // +inf: no key either, as merge_attn_states reads it
      const float mx = fmaxf(prior, lse);
      if (lse == -INFINITY) continue;   // nothing visible here: the row stands
      const float wp = prior == -INFINITY ? 0.f : __expf(prior - mx), wn = __expf(lse - mx);
      const float tot = wp + wn, other = wp / tot;
      mul *= wn / tot;
      u32x2 old[DPL];
#pragma unroll
      for (int i = 0; i < DPL; ++i) old[i] = *reinterpret_cast<const u32x2*>(op + 16 * i + 4 * g_end);
#pragma unroll
      for (int i = 0; i < DPL; ++i) {
        float f[4];
        unpack2<DT>(old[i].x, f[0], f[1]);
        unpack2<DT>(old[i].y, f[2], f[3]);
        u32x2 w;
        w.x = pack2<DT>(__builtin_fmaf(f[0], other, oacc[rb][i][0] * mul), __builtin_fmaf(f[1], other, oacc[rb][i][1] * mul));
        w.y = pack2<DT>(__builtin_fmaf(f[2], other, oacc[rb][i][2] * mul), __builtin_fmaf(f[3], other, oacc[rb][i][3] * mul));
        *reinterpret_cast<u32x2*>(op + 16 * i + 4 * g_end) = w;
      }
      if (g_end == 0) *lp = __logf(tot) + mx;
      continue;
    }
    // block i: the lane holds dims 16 i + 4 g .. + 3 of its row
#pragma unroll
    for (int i = 0; i < DPL; ++i) {
      u32x2 w;
      w.x = pack2<DT>(oacc[rb][i][0] * mul, oacc[rb][i][1] * mul);
      w.y = pack2<DT>(oacc[rb][i][2] * mul, oacc[rb][i][3] * mul);
      *reinterpret_cast<u32x2*>(op + 16 * i + 4 * g_end) = w;
    }
    if (a.lse != nullptr && g_end == 0) a.lse[(int64_t)head * a.total_q + tok] = lse;
  }
}

// How many of an XCD's last pairs a causal launch takes block by block: those of two rounds of workgroups, or none.  `live`
// counts the workgroups that have rows, as far as the host knows.  What the order changes, the launch alone, us on MI355X,
// pair by pair / so:
//   up to one live workgroup per compute unit there is no second round to even out, and a pair's blocks side by side find its
//   keys in L2: 16 heads, requests of 490 and 1190 tokens (224 live) 36.9 / 38.2, of 1700 and 300 (256) 49.8 / 53.0, of 2000
//   (256) 55.7 / 55.7; but 16 heads x 2560 (336) 75.8 / 74.1, 20 x 2000 (320) 73.6 / 58.8, 32 x 1280 (352) 46.5 / 43.0, 64 x 1000
//   (512) 45.4 / 38.7, 128 x 1000 (1024) 76.8 / 63.2, 128 heads, 4 requests of 430 - 1220 (2944) 156.6 / 149.1;
//   up to three blocks hardly differ in length: 128 heads, 4 of 200 28.8 / 30.1, 4 of 300 44.5 / 47.3, 64 heads, 8 of 380
//   56.2 / 56.4; with four 128 heads, 4 of 500 96.7 / 83.7, 16 heads, 8 of 500 30.0 / 26.1;
//   where most of the grid has no rows, a long request's blocks lie a fixed number of places apart and pile up on part of an
//   XCD (with the places rotated from block to block they do not); two rounds of live ones even that out.  16 heads, 7 of
//   100 and one of 1500 (336 live of 1536) 47.7 / 66.2, but 7 of 100 and one of 3000 (512 of 3072) 104.9 / 99.5, 32 heads, 4 of
//   150 and one of 1300 (544 of 1760) 63.2 / 50.5, 15 of 100 and one of 2000 (1120 of 8192) 104.1 / 95.3.
static int by_block_pairs(dim3 grid, int64_t live, int max_seqlen_q, int64_t total_q) {
  const int64_t units = num_cus();
  const bool half_live = 2 * total_q >= (int64_t)max_seqlen_q * grid.z;
  if (grid.x < 4 || live <= units || !(half_live || live >= 2 * units)) return 0;
  const unsigned pairs = grid.y * grid.z, bits = xcd_bits_of(pairs);
  const int64_t last = ((2 * kPerUnit * units) >> bits) / grid.x + 1;
  return (int)(last < (pairs >> bits) ? last : (pairs >> bits));
}

template <int NOPE, int ROPE, int DV>
static int launch_varlen(int dtype, const VarlenArgs& args, int max_seqlen_q, dim3 grid, hipStream_t s) {
  VarlenArgs a = args;
  // the lengths are device data; rows and sequences give the number of workgroups to within half of one per sequence
  const int64_t live = (a.total_q / 128 + (grid.z + 1) / 2) * (int64_t)grid.y;
  a.last_pairs = a.causal ? by_block_pairs(grid, live, max_seqlen_q, a.total_q) : 0;
  if (dtype == KVQ_F16) hipLaunchKernelGGL((varlen_attn_kernel<KVQ_F16, NOPE, ROPE, DV>), grid, dim3(256), 0, s, a);
  else hipLaunchKernelGGL((varlen_attn_kernel<KVQ_BF16, NOPE, ROPE, DV>), grid, dim3(256), 0, s, a);
  return check_hip(hipGetLastError(), "mla_prefill_attn launch");
}

}  // namespace kvq

extern "C" int kvq_mla_prefill_attn(const void* q, int dtype, int64_t q_stride_tok, int64_t q_stride_head,
                                    const void* k_nope, int64_t kn_stride_tok, int64_t kn_stride_head,
                                    const void* k_pe, int64_t kpe_stride_tok, const void* v, int64_t v_stride_tok,
                                    int64_t v_stride_head, const int32_t* cu_seqlens_q, const int32_t* cu_seqlens_k,
                                    int num_seqs, int max_seqlen_q, int64_t total_q, int num_heads, int nope_dim,
                                    int rope_dim, int v_dim, float scale, int causal, void* out,
                                    int64_t out_stride_tok, int64_t out_stride_head, float* lse,
                                    kvq_stream_t stream) {
  using namespace kvq;
  const char* op = "mla_prefill_attn";
  KVQ_REQUIRE(num_seqs >= 0 && max_seqlen_q >= 0 && total_q >= 0 && num_heads > 0, "%s: bad sizes", op);
  if (num_seqs == 0 || max_seqlen_q == 0 || total_q == 0) return KVQ_OK;
  KVQ_REQUIRE(dtype == KVQ_BF16 || dtype == KVQ_F16, "%s: q, k and v must be bf16 or fp16 (dtype %d)", op, dtype);
  KVQ_REQUIRE(scale > 0.f && scale < INFINITY, "%s: scale must be positive and finite", op);   // the kernel takes row maxima before scaling
  KVQ_REQUIRE(q && k_nope && v && out && cu_seqlens_q && cu_seqlens_k, "%s: NULL pointer", op);
  KVQ_REQUIRE((causal & ~(KVQ_MLA_PREFILL_CAUSAL | KVQ_MLA_PREFILL_MERGE)) == 0, "%s: unknown flag in causal (%d)", op, causal);
  KVQ_REQUIRE(!(causal & KVQ_MLA_PREFILL_MERGE) || lse != nullptr, "%s: the state to merge into has no lse", op);
  KVQ_REQUIRE(rope_dim == 0 || k_pe != nullptr, "%s: k_pe is NULL with rope_dim %d", op, rope_dim);
  KVQ_REQUIRE(num_heads <= 65535 && num_seqs <= 65535, "%s: more than 65535 heads or sequences", op);
  const int64_t strides[] = {q_stride_tok, q_stride_head, kn_stride_tok, kn_stride_head, kpe_stride_tok,
                             v_stride_tok, v_stride_head, out_stride_tok, out_stride_head};
  for (int64_t st : strides) KVQ_REQUIRE(st >= 0 && st % 8 == 0, "%s: strides must be multiples of 8 elements (got %lld)", op, (long long)st);
  // a tile's 32 rows are addressed with 32-bit offsets from its first key
  KVQ_REQUIRE(kn_stride_tok < (1 << 24) && kpe_stride_tok < (1 << 24) && v_stride_tok < (1 << 24),
              "%s: token strides must be below 2^24 elements", op);
  KVQ_REQUIRE(((uintptr_t)q | (uintptr_t)k_nope | (uintptr_t)k_pe | (uintptr_t)v | (uintptr_t)out) % 16 == 0,
              "%s: tensors must be 16-byte aligned", op);
  VarlenArgs a{};
  a.q = q; a.k_nope = k_nope; a.k_pe = rope_dim ? k_pe : k_nope; a.v = v; a.out = out; a.lse = lse;
  a.cu_q = cu_seqlens_q; a.cu_k = cu_seqlens_k;
  a.q_st = q_stride_tok; a.q_sh = q_stride_head; a.kn_st = kn_stride_tok; a.kn_sh = kn_stride_head;
  a.kpe_st = kpe_stride_tok; a.v_st = v_stride_tok; a.v_sh = v_stride_head;
  a.out_st = out_stride_tok; a.out_sh = out_stride_head; a.total_q = total_q;
  a.causal = (causal & KVQ_MLA_PREFILL_CAUSAL) != 0;
  a.merge = (causal & KVQ_MLA_PREFILL_MERGE) != 0;
  a.scale_log2 = scale * kLog2e;
  const dim3 grid((unsigned)((max_seqlen_q + 127) / 128), (unsigned)num_heads, (unsigned)num_seqs);
  hipStream_t s = as_stream(stream);
  if (nope_dim == 128 && rope_dim == 64 && v_dim == 128) return launch_varlen<128, 64, 128>(dtype, a, max_seqlen_q, grid, s);
  if (nope_dim == 64 && rope_dim == 32 && v_dim == 64) return launch_varlen<64, 32, 64>(dtype, a, max_seqlen_q, grid, s);
  if (nope_dim == 128 && rope_dim == 0 && v_dim == 128) return launch_varlen<128, 0, 128>(dtype, a, max_seqlen_q, grid, s);
  return fail(KVQ_EINVAL, "%s: head dims (nope %d, rope %d, v %d) are not built; built: (128, 64, 128), (64, 32, 64), (128, 0, 128)",
              op, nope_dim, rope_dim, v_dim);
}
