// The workgroup-shared prefill tile: long query runs over the paged cache, the compute-bound shape (gfx950).
//
// Four waves of 32 columns -- (query token, q head) pairs -- share one kv head's 32-token tiles.  A tile's records stream
// from memory straight into LDS, are expanded ONCE per workgroup to fp16 -- K as [8-dim chunk][token], V transposed as
// [8-token chunk][dim], both with the code bias taken out, so that every operand of the products is one 16-byte LDS read
// at a constant offset -- and each wave runs S^T = K Q^T, the softmax and O^T += V^T P~ of its columns on the 32x32x16
// MFMA.  A lane holds 16 tokens of ONE column.
//
// What bounds it.  With two workgroups on a compute unit, latency: every unit about half busy (counters: matrix unit 36 %,
// LDS 50 %, vector unit 45 %).  So the plain kernel is built for THREE workgroups per compute unit, 168 registers and 50 KB
// of LDS each, which is what the rest follows from: tiles go from memory into LDS without passing through registers, the
// operands of a tile are read as they are used up, a token's scales reach the lanes by a broadcast inside the multiply
// (one LDS read per tile instead of four 16-byte ones) and a wave loads from one half tile only (one block table entry, one
// resource).  168 registers hold what a step needs and no more: lane number, column and limit, which only the masked steps
// and the ends of the walk use, are worked out anew there.  Kept through the loops they were spilled, 11 to 14 of them, and
// some reloaded in every step behind the next tile's loads, which the reload then waited for (16 prompts of 300 tokens 60.1
// -> 54.5 us, one of 2000 82.9 -> 74.0, the mixed step below 447 -> 437).  One value is left, spilled outside the loops; head
// size 64 spills up to three with the extras, at head size 128 those do not spill.  At three workgroups the vector unit is 65 % busy, the matrix unit 45 %, the LDS 51 %.
// Measured on MI355X against two workgroups per compute unit with register loads and padded tiles: 4 x 2048 new tokens on
// 0-6k cached ones beside 60 decode rows (28/4 heads) 534 -> 442 us for the step, 512 tokens on 32k in context ranges (32/8 heads)
// 395 -> 341 us; captured: a 2000-token prompt 98.7 -> 74.0 us, with int4 codes 103.7 -> 79.7, head size 64 77.4 -> 60.5, one of 70
// tokens 15.8 -> 14.0, a window of 1500 tokens in the mixed step 320 -> 271, with a soft cap 736 -> 653.
// One wave per SIMD with 64 columns each (half the operand reads and expansion work) reached 334 us for the 512 tokens,
// but 497 us for the mixed step: a wave alone issues an instruction every 5.6 cycles, two or more waves one every 2 to 4.
#pragma once

#include "kvq_prefill_impl.cuh"

namespace kvq {

typedef float floatx16 __attribute__((ext_vector_type(16)));

template <int D, int CODE>
struct SharedTile {
  using DTile = DecodeTile<D, KVQ_BF16, KVQ_BF16, CODE>;
  static constexpr bool FP8 = DTile::FP8;     // e4m3fn codes: they enter the MFMA as value / 2^8, without a bias
  static constexpr bool INT4 = DTile::INT4;   // two codes per byte
  static constexpr int DB = DTile::DB;        // code bytes of a half record
  static constexpr int WAVES = 4;
  static constexpr int COLS = 32 * WAVES;
  static constexpr int KS = D / 16, MT = D / 32;   // k-steps of the QK product, 32-dim row tiles of O^T
  static constexpr int NCH = 2 * DB / 16;          // whole 16-byte chunks of a record; its last 8 bytes are kept apart
  static constexpr int ROWS = 64 / NCH;            // records a wave's load covers
  static constexpr int LOADS = 16 / ROWS > 2 ? 16 / ROWS / 2 : 1;  // chunk loads per wave and tile
  // raw tile: [32 records][NCH chunks, chunk c of record r in slot c ^ (r % NCH)], then per 16-token half the records'
  // last 8 bytes (256 bytes per half: the loads that bring them write 64 dwords, the second 32 a copy of the first)
  static constexpr int RAW_ROW = 16 * NCH, RAW_TAIL = kTile * RAW_ROW, RAW_BYTES = RAW_TAIL + 512;
  static constexpr int K_BYTES = kTile * D * 2, V_BYTES = kTile * D * 2;
  static constexpr int SC_BYTES = 68 * 4;          // 32 K-side and 32 V-side scales, the tile's lazy-maximum allowance
  static constexpr int BUF_BYTES = K_BYTES + V_BYTES + SC_BYTES;
  static constexpr int LDS_BYTES = 2 * RAW_BYTES + 2 * BUF_BYTES;

  // A wave's share of a 16-token half, straight into LDS: lane i's 16 (tail: 4) bytes land at dst + 16 i (tail + 4 i).
  __device__ static __forceinline__ void load_half(__amdgpu_buffer_rsrc_t w, uint32_t offset, const uint32_t (&g_chunk)[LOADS],
                                                   uint32_t g_tail, uint8_t* dst, uint8_t* tail) {
    typedef __attribute__((address_space(3))) void* lds_ptr_t;
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(w, (lds_ptr_t)(dst + i * 1024), 16, g_chunk[i], offset, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(w, (lds_ptr_t)tail, 4, g_tail, offset, 0, 0);
  }

  // ---- expansion -------------------------------------------------------------------------------------------------
  // Byte `at` of record r in the raw tile.
  __device__ static __forceinline__ uint32_t raw_at(int r, int at) {
    return at < RAW_ROW ? (uint32_t)(r * RAW_ROW + (((at >> 4) ^ (r & (NCH - 1))) << 4) + (at & 15))
                        : (uint32_t)(RAW_TAIL + (r >> 4) * 256 + (r & 15) * 8 + (at - RAW_ROW));
  }
  // A thread converts 16 code bytes of one token's K and a 4-token x 4-dim block of V; what it reads and writes:
  struct Places {
    uint32_t k_raw, k_out, v_raw[4], v_out, sc_raw;
  };
  // 16 neighbouring lanes read one K chunk of 16 records (16 slots, no bank twice) and write 256 bytes in a row; 32
  // neighbouring lanes read 32 dwords in a row of a V record.  A wave's two V blocks of four tokens are the two that
  // share the 16-byte pieces of the expanded V.
  __device__ static __forceinline__ Places places(int tid) {
    constexpr int KCH = DB / 16, QB = INT4 ? 2 : 4;   // K chunks per record; bytes of four V codes
    Places p;
    const int tok = tid % kTile, ch = (tid / kTile) % KCH;
    p.k_raw = raw_at(tok, 16 * ch);
    p.k_out = (uint32_t)(ch * (INT4 ? 4 : 2) * 512 + tok * 16);
    const int dq = tid % (D / 4), idx = (tid / (D / 4)) & 7;
    const int tg = (idx & 4) | ((idx & 1) << 1) | ((idx >> 1) & 1);   // tokens 4 tg .. 4 tg + 3
#pragma unroll
    for (int a = 0; a < 4; ++a) p.v_raw[a] = raw_at(4 * tg + a, DB + 4 + QB * dq);
    // token t of the tile sits at position (t/16)*16 + ((t%8)/4)*8 + ((t/8)%2)*4 + t%4: the order in which the 32x32
    // accumulator of S^T hands a lane its tokens
    const int chunk = 2 * (tg >> 2) + (tg & 1), half = (tg >> 1) & 1;
    p.v_out = (uint32_t)(K_BYTES + chunk * D * 16 + dq * 16 + half * 8);
    const int lane = tid & 63;
    p.sc_raw = raw_at(lane & 31, lane < 32 ? DB : 2 * DB + 4);
    return p;
  }
  struct Expand {
    u32x4 w;
    uint32_t t[4];
    uint32_t a01, b01, a23, b23;
    float sc;
  };
  __device__ static __forceinline__ void expand_load(Expand& e, const Places& p, const uint8_t* raw) {
    e.w = *reinterpret_cast<const u32x4*>(raw + p.k_raw);
    e.sc = *reinterpret_cast<const float*>(raw + p.sc_raw);
#pragma unroll
    for (int a = 0; a < 4; ++a) {
      if constexpr (INT4) e.t[a] = *reinterpret_cast<const uint16_t*>(raw + p.v_raw[a]);
      else e.t[a] = *reinterpret_cast<const uint32_t*>(raw + p.v_raw[a]);
    }
  }
  // Two code bytes / two nibbles of y (= codes ^ 0x88...) as two fp16 codes, bias taken out.
  template <bool GARBAGE>
  __device__ static __forceinline__ uint32_t to_half2(uint32_t x, bool upper) {
    if constexpr (FP8) return fp8_bytes_to_half2<GARBAGE>(x, upper);
    const half2_t bias = {(half_t)kCodeBias, (half_t)kCodeBias};
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, bytes_to_half2(x, upper)) - bias);
  }
  __device__ static __forceinline__ uint32_t nibbles_to_codes(uint32_t y, int k) {
    const half2_t bias = {(half_t)kCodeBiasInt4, (half_t)kCodeBiasInt4};
    return __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, nibbles_to_half2(y, k)) - bias);
  }
  // The expansion in pieces, four for K and five for V, each for a place between two products.
  __device__ static __forceinline__ void expand_k_piece(Expand& e, const Places& p, int i, uint8_t* buf) {
    if constexpr (INT4) {   // the and-or conversion yields dims 0 4 1 5 2 6 3 7 of a dword
      const uint32_t y = e.w[i] ^ 0x88888888u;
      const uint32_t h0 = nibbles_to_codes(y, 0), h1 = nibbles_to_codes(y, 1);
      const uint32_t h2 = nibbles_to_codes(y, 2), h3 = nibbles_to_codes(y, 3);
      u32x4 o;
      o.x = perm(h1, h0, kPermLowHalves);
      o.y = perm(h3, h2, kPermLowHalves);
      o.z = perm(h1, h0, kPermHighHalves);
      o.w = perm(h3, h2, kPermHighHalves);
      *reinterpret_cast<u32x4*>(buf + p.k_out + 512 * i) = o;
    } else {
      const uint32_t x = prep_codes<FP8>(e.w[i]);
      const uint32_t a = to_half2<false>(x, false), b = to_half2<false>(x, true);
      if ((i & 1) == 0) {
        e.a01 = a;
        e.b01 = b;
      } else {
        *reinterpret_cast<u32x4*>(buf + p.k_out + 512 * (i >> 1)) = (u32x4){e.a01, e.b01, a, b};
      }
    }
  }
  // GARBAGE: the tile may hold slots past the end of the sequence or below the window.
  template <bool GARBAGE>
  __device__ static __forceinline__ void expand_v_piece(Expand& e, const Places& p, int i, uint8_t* buf) {
    if (i == 0) {
      if constexpr (INT4) {
        e.a01 = (e.t[0] | (e.t[1] << 16)) ^ 0x88888888u;
        e.a23 = (e.t[2] | (e.t[3] << 16)) ^ 0x88888888u;
      } else {
#pragma unroll
        for (int a = 0; a < 4; ++a) e.t[a] = prep_codes<FP8>(e.t[a]);
        e.a01 = perm(e.t[1], e.t[0], 0x05010400u);
        e.b01 = perm(e.t[1], e.t[0], 0x07030602u);
        e.a23 = perm(e.t[3], e.t[2], 0x05010400u);
        e.b23 = perm(e.t[3], e.t[2], 0x07030602u);
      }
      return;
    }
    const int b = i - 1;
    u32x2 o;
    if constexpr (INT4) {
      o.x = nibbles_to_codes(e.a01, b);
      o.y = nibbles_to_codes(e.a23, b);
    } else {
      o.x = to_half2<GARBAGE>(b < 2 ? e.a01 : e.b01, b & 1);
      o.y = to_half2<GARBAGE>(b < 2 ? e.a23 : e.b23, b & 1);
    }
    *reinterpret_cast<u32x2*>(buf + p.v_out + b * (D / 4) * 16) = o;   // dim 4 dq + b is row b D/4 + dq
  }
  // The lane number, worked out anew (kept from tile to tile it, and what follows from it, were spilled).
  __device__ static __forceinline__ uint32_t lane_anew() {
    uint32_t lane;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
    return lane;
  }
  // The tile's scales; one wave does it.
  __device__ static __forceinline__ void expand_scales(float sc, uint8_t* buf, float k_mul) {
    const uint32_t lane = lane_anew();
    const float sc_mul = lane < 32 ? k_mul : kPScale;
    // a slot that holds no token: anything, made finite; the softmax scale, and with it the K side, may be negative
    const float val = fminf(fmaxf(sc * sc_mul, -65504.f), 65504.f);
    float* out = reinterpret_cast<float*>(buf + K_BYTES + V_BYTES);
    out[lane] = val;
    // how far a logit may exceed a column's reference maximum in this tile before the maximum has to move:
    // 2^kLazyMax * (largest V-side scale) must stay inside fp16, else nothing is allowed
    const bool any_big = __builtin_amdgcn_ballot_w64(lane >= 32 && val > kLazyScaleMax) != 0;
    out[64 + (lane & 3)] = any_big ? 0.f : kLazyMax;
  }

  // The value that lane n of the lane's row of 16 holds (folded into the instruction that uses it).
  __device__ static __forceinline__ float row_lane(float v, int n) {
    switch (n) {
#define KVQ_ROW_LANE(N) case N: return as_f32(__builtin_amdgcn_update_dpp(0, as_u32(v), 0x150 + N, 0xf, 0xf, true))
      KVQ_ROW_LANE(0); KVQ_ROW_LANE(1); KVQ_ROW_LANE(2); KVQ_ROW_LANE(3); KVQ_ROW_LANE(4); KVQ_ROW_LANE(5); KVQ_ROW_LANE(6); KVQ_ROW_LANE(7);
      KVQ_ROW_LANE(8); KVQ_ROW_LANE(9); KVQ_ROW_LANE(10); KVQ_ROW_LANE(11); KVQ_ROW_LANE(12); KVQ_ROW_LANE(13); KVQ_ROW_LANE(14);
      default: KVQ_ROW_LANE(15);
#undef KVQ_ROW_LANE
    }
  }

  // Products -> logits (in place), masked; returns the lane's largest.  ksc: lane n of a row of 16 holds the K scale of
  // the token in register n.
  template <bool MASK, bool EXT>
  __device__ static __forceinline__ float logits(float ksc, const AttnIO& io, float ali, int limit, uint32_t wspan, int t,
                                                 int lane, bool biased, floatx16& s) {
    const int tok0 = t * kTile + 4 * (lane >> 5);
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] *= row_lane(ksc, i);
    if constexpr (EXT) {
      if (io.cap_c != 0.f) {
        float x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) x[i] = s[i];
        soft_cap(x, io.cap_c, io.cap_k);
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = x[i];
      }
      if (biased) {
        const float rel = (float)(tok0 - (limit - 1));
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = __builtin_fmaf(ali, rel + (float)((i >> 2) * 8 + (i & 3)), s[i]);
      }
    }
    float d = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      if constexpr (MASK) {
        const int tok = tok0 + (i >> 2) * 8 + (i & 3);
        if constexpr (EXT) s[i] = ((uint32_t)(limit - 1 - tok) < wspan) ? s[i] : -INFINITY;
        else s[i] = (tok < limit) ? s[i] : -INFINITY;
      }
      d = fmaxf(d, s[i]);
    }
    return d;
  }

  // V^T row b D/4 + q of the expanded tile is dim 4 q + b, so row r of the accumulators (register 4 (r / 8) + r % 4 of
  // half (r / 4) % 2) is that dim: a lane holds D / 8 runs of four dims, run i's dim b being row b D/4 + 4 g + its q.
  __device__ static constexpr int run_row(int i) { return (i / 4) * 8 + i % 4; }
  __device__ static __forceinline__ float o_dim(const floatx16 (&o)[MT], int i, int b) {
    const int r = b * (D / 4) + run_row(i);
    return o[r / 32][((r % 32) / 8) * 4 + r % 4];
  }
  // Two floats in bf16: the bits of f32_to_bf16_bits, by selects (its early return became two branches per element, and an
  // epilogue of 2300 instructions that a short prompt's launch fetched for the first time).
  __device__ static __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    auto upper = [](float f) {
      const uint32_t u = as_u32(f), rounded = u + 0x7fffu + ((u >> 16) & 1u);
      return (u & 0x7fffffffu) > 0x7f800000u ? (u | 0x400000u) : rounded;
    };
    return perm(upper(hi), upper(lo), kPermHighHalves);
  }
  __device__ static __forceinline__ int first_dim(int i, int g) { return 4 * (run_row(i) + 4 * g); }

  // Q of the lane's column as the second operand: lane (c = lane & 31, g = lane >> 5) holds, for k-step ks, dims
  // 16 ks + 8 g + j, rounded to fp16 (exact for bf16 values in fp16's range).
  template <int QDT>
  __device__ static __forceinline__ void load_q(const AttnIO& io, int64_t elem, bool valid, int lane, half8_t (&qb)[KS]) {
    constexpr int N = QDT == KVQ_F32 ? 2 : 1;
    const uint32_t okmask = valid ? 0xffffffffu : 0u;
    const int64_t first = elem + 8 * (lane >> 5);
    u32x4 raw[KS][N];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int i = 0; i < N; ++i)
        raw[ks][i] = *reinterpret_cast<const u32x4_a4*>(static_cast<const uint8_t*>(io.q) + (first + 16 * ks) * (2 * N) + 16 * i);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      u32x4 hb;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        float lo, hi;
        if constexpr (QDT == KVQ_F32) {
          const uint32_t x = raw[ks][w >> 1][2 * (w & 1)], y = raw[ks][w >> 1][2 * (w & 1) + 1];
          lo = as_f32(x);
          hi = as_f32(y);
        } else {
          const uint32_t x = raw[ks][0][w];
          if constexpr (QDT == KVQ_BF16) {
            lo = as_f32(x << 16);
            hi = as_f32(x & 0xffff0000u);
          } else {
            const half2_t h = __builtin_bit_cast(half2_t, x);
            lo = (float)h.x;
            hi = (float)h.y;
          }
        }
        hb[w] = pack_half2(clamp_half_range(lo), clamp_half_range(hi)) & okmask;
      }
      qb[ks] = __builtin_bit_cast(half8_t, hb);
    }
  }
};

// The sequence of workgroup `lin` of a launch with `per_seq` workgroups per query run (-1: there are not as many runs),
// longest sequence first: workgroups start in this order, and the longest sequence's are the ones that should not start last.
// Up to kRunsInKernel sequences: a lane for each, one trip to memory, ranked by lane moves inside the row of 16.  With the
// plan kernel in front of them too, a step with a prompt of 70 tokens (32/8 heads of 128) took 14.0 us for 12.0, one of 2000
// 71.7 for 69.2.  Beyond, and for the per-wave tile, the plan kernel lists them once: ranked in every workgroup, 64 prompts of
// 200 - 400 tokens took 193 us for 180.
// (PLANNED: an instantiation of its own, since choosing at run time cost launches with a plan up to 1 %.)
template <bool PLANNED>
__device__ __forceinline__ int find_run(const PrefillArgs& a, unsigned lin, unsigned per_seq) {
  if constexpr (PLANNED) {
    return lin >= per_seq * (unsigned)a.plan[0] ? -1 : a.plan[1 + lin / per_seq];
  }
  static_assert(kRunsInKernel == 16, "a lane of one row for every sequence");
  const int lane = threadIdx.x & 63, s = min(lane, a.num_seqs - 1);
  const int q_len = a.cu_seqlens_q[s + 1] - a.cu_seqlens_q[s], len = a.seq_lens[s];
  const bool has = lane < a.num_seqs && q_len > 1 && len > 0;
  if (lin >= per_seq * (unsigned)__builtin_popcountll(__builtin_amdgcn_ballot_w64(has))) return -1;
  // distinct; of sequences of the same length the first
  const uint32_t key = has ? (uint32_t)min(len, (1 << 27) - 1) * 16u + (uint32_t)(15 - lane) : 0u;
  unsigned rank = 0;
#define KVQ_RANK(N) rank += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)key, 0x120 + N, 0xf, 0xf, true) > key ? 1u : 0u;   // row_ror:N
  KVQ_RANK(1) KVQ_RANK(2) KVQ_RANK(3) KVQ_RANK(4) KVQ_RANK(5) KVQ_RANK(6) KVQ_RANK(7) KVQ_RANK(8)
  KVQ_RANK(9) KVQ_RANK(10) KVQ_RANK(11) KVQ_RANK(12) KVQ_RANK(13) KVQ_RANK(14) KVQ_RANK(15)
#undef KVQ_RANK
  return __builtin_ctzll(__builtin_amdgcn_ballot_w64(has && rank == lin / per_seq));
}

// EXT adds the sliding window, the logits soft cap and ALiBi; the plain causal kernel carries none of them.
// With a.ksplit > 1 the grid's x dimension carries that many context ranges per query block; a workgroup takes one range
// of its item's tiles and writes a partial state instead of the rows.
// Waves per SIMD: the extras need 190 registers at head size 128 (at 168 they spill inside the loop: a window of 2000
// tokens 331 us against 285), head size 64 fits 128 (mixed batch 264 us at three waves, 255 at four; with a soft cap 314 at three,
// 358 at four, but with a window alone 129 and 120).
template <int D, bool EXT>
constexpr int kSharedWaves = D == 64 ? 4 : EXT ? 2 : 3;

template <int D, bool EXT, int CODE, bool PLANNED>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(kSharedWaves<D, EXT>, kSharedWaves<D, EXT>)))
void paged_prefill_shared_kernel(PrefillArgs a, int q_dtype, int out_dtype) {
  using W = SharedTile<D, CODE>;
  using DTile = typename W::DTile;
  constexpr int KS = W::KS, MT = W::MT;
  __shared__ __align__(16) uint8_t lds[W::LDS_BYTES];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Which sequence, kv head and query block this workgroup takes.  Workgroups start in the order of their linear
  // number and go to the eight XCDs in turn by it.  The number is read over the sequences that HAVE a query run
  // (find_run; the surplus workgroups of the grid, which is sized for every sequence of the batch, come last and
  // leave at once), sequence by sequence, and inside a sequence query-block-major over its kv heads, longest block
  // first: the heads of a sequence then walk the same tokens at the same time (their records are neighbours in
  // memory, and what one head's workgroup brought into L2 is there for the next), and the head is shifted by the
  // block number so that a head's blocks visit every XCD in turn.  Measured against the grid read as launched
  // (block, sequence, head): the mixed batch of 4 x 2048 new tokens 852 -> 752 us per attention call, one
  // 8192-token prompt 908 -> 733 us, 16 prompts of 1024 tokens 410 -> 291 us (there XCD 0 had the longest block
  // of every eight of every pair), 4 x 1024 new tokens on 8k-32k cached ones 2.43 -> 2.02 ms.  Query-block-major
  // over ALL pairs was better still for short prompts from scratch (16 x 512: 103 against 113 us) and much worse
  // with long contexts (the mixed batch 959 us: sixteen streams of keys at once, six times the HBM fetches).
  const unsigned nsplit = (unsigned)a.ksplit;
  const unsigned nqb = gridDim.x / nsplit, hk = gridDim.z, per_seq = nqb * hk;
  const unsigned lin_all = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
  const unsigned lin = lin_all / nsplit;
  const int seq = find_run<PLANNED>(a, lin, per_seq);
  if (seq < 0) return;   // uniform over the workgroup
  unsigned split = lin_all % nsplit;   // the splits of an item are neighbours in launch order
  const unsigned rem = lin % per_seq;
  int qb = (int)(rem / hk);
  int hkv = (int)((rem % hk + (unsigned)qb) % hk);
  // Context ranges: all query blocks of a (kv head, range) pair go to ONE XCD, whose L2 then serves the range's records to
  // all but the first of them, where the pairs can be dealt out to the eight evenly (512 tokens on 32k, 8 kv heads, 6 ranges:
  // a step 388 -> 366 us, 1000 on 50k 1097 -> 1032, 4 kv heads 352 -> 342).
  if (nsplit > 1 && nqb > 1 && (hk * nsplit & 7) == 0) {
    const unsigned r = lin_all % (per_seq * nsplit), k = r >> 3, pair = k / nqb * 8 + (r & 7);
    qb = (int)(k % nqb);
    hkv = (int)(pair % hk);
    split = pair / hk;
  }
  const AttnIO& io = a.io;
  const int q_begin = a.cu_seqlens_q[seq];
  const int q_len = a.cu_seqlens_q[seq + 1] - q_begin;
  const int len = a.seq_lens[seq];
  const int q0 = ((int)nqb - 1 - qb) * a.q_tokens;
  if (q_len <= 1 || q0 >= q_len || len <= 0) return;   // uniform over the workgroup
  if (a.route == 1 && q_len * io.group < 64) return;    // the per-wave tile's

  // column of a lane: (query token q0 + n / group, head n % group), n = wave * 32 + (lane & 31); n / group by a
  // reciprocal: both are small, and n + 1/2 is half a column away from every multiple
  const int ctx = len - q_len;
  struct Column {
    bool valid;
    int qi, head;
    int64_t row;
  };
  const float per_column = as_f32(__builtin_amdgcn_readfirstlane(as_u32(__builtin_amdgcn_rcpf((float)io.group))));
  auto column = [&](int of_lane) __attribute__((always_inline)) {
    const int n = wave * 32 + (of_lane & 31);
    const int qt = (int)(((float)n + 0.5f) * per_column);
    Column c;
    c.qi = q0 + qt;
    c.valid = qt < a.q_tokens && c.qi < q_len;
    c.head = hkv * io.group + (n - qt * io.group);
    c.row = q_begin + (c.valid ? c.qi : q0);
    return c;
  };
  auto limit_of = [&](const Column& c) __attribute__((always_inline)) {
    const int lim = a.causal ? ctx + c.qi + 1 : len;
    return c.valid ? (lim < 0 ? 0 : (lim > len ? len : lim)) : 0;
  };
  const Column col = column(lane);
  int limit = limit_of(col), step_lane = lane;   // of the masked steps
  const int wave_max_limit = wave_max_i32(limit);
  const int wave_min_limit = -wave_max_i32(col.valid ? -limit : -0x7fffffff);
  int wg_limit = a.causal ? ctx + min(q0 + a.q_tokens, q_len) : len;
  wg_limit = wg_limit < 0 ? 0 : (wg_limit > len ? len : wg_limit);
  const int t_end = (wg_limit + kTile - 1) / kTile;
  // Sliding window: a column sees [limit - window, limit).  The workgroup starts at the (even) tile that holds the first
  // query token's lower edge; a wave masks tiles below the latest lower edge among its columns.
  uint32_t wspan = 0x7fffffffu;
  int t_first = 0, wg_first = 0, wave_max_first = 0;
  if constexpr (EXT) {
    if (io.window > 0) {
      wspan = (uint32_t)io.window;
      wg_first = max(0, (a.causal ? ctx + q0 + 1 : len) - io.window);
      t_first = (wg_first / kTile) & ~1;
      wave_max_first = max(0, wave_max_limit - io.window);
    }
  }

  floatx16 o[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int i = 0; i < 16; ++i) o[mt][i] = 0.f;
  float m = 0.f, l = 0.f;   // reference maximum (of account once the column has seen a token), lane's sum of weights
  bool seen = false;

  // this workgroup's tiles: all of the item's, or one of nsplit ranges of an even number of tiles
  const int per = (((t_end - t_first) + (int)nsplit - 1) / (int)nsplit + 1) & ~1;
  const int t_lo = t_first + (int)split * per;
  const int t_hi = min(t_end, t_lo + per);
  if (t_hi > t_lo) {
    // ---- loads.  A wave brings chunks of ONE 16-token half of every tile, and the last 8 bytes of that half's records:
    // one block table entry and one resource per tile.  The place in the cache is stepped by additions; past the
    // sequence's last block the last one is read again (and masked).
    const int32_t* bt_row = io.block_table + (int64_t)seq * io.bt_stride;
    const int half = wave & 1;
    const uint32_t ss = (uint32_t)io.g.stride_slot, blk_bytes = (uint32_t)io.g.block_size * ss;
    const int last_entry = DTile::div_bs(io, len + io.g.block_size - 1) - 1;
    const uint8_t* const cache_head = io.cache + io.g.k_off + (uint64_t)((uint32_t)hkv * (uint32_t)io.g.stride_head);
    const int step_entries = kTile / io.g.block_size;
    const uint32_t step_bytes = (uint32_t)(kTile - step_entries * io.g.block_size) * ss;
    int entry = DTile::div_bs(io, t_lo * kTile + 16 * half);
    uint32_t in_block = (uint32_t)DTile::mod_bs(io, t_lo * kTile + 16 * half) * ss;
    int32_t block;
    uint32_t offset;
    auto next_place = [&]() __attribute__((always_inline)) {
      block = *reinterpret_cast<const_i32_ptr>(reinterpret_cast<uintptr_t>(bt_row) + 4u * (uint32_t)min(entry, last_entry));
      offset = in_block;
      in_block += step_bytes;
      const bool over = in_block >= blk_bytes;
      in_block -= over ? blk_bytes : 0u;
      entry += step_entries + (over ? 1 : 0);
    };
    const int first_row = ((wave >> 1) * W::LOADS * W::ROWS) & 15;   // of the half (one load may cover it: then two waves bring the same)
    uint32_t g_chunk[W::LOADS];
#pragma unroll
    for (int i = 0; i < W::LOADS; ++i) {
      const int r = first_row + i * W::ROWS + lane / W::NCH;
      g_chunk[i] = (uint32_t)r * ss + 16u * (uint32_t)((lane % W::NCH) ^ ((16 * half + r) & (W::NCH - 1)));
    }
    const uint32_t g_tail = (uint32_t)((lane & 31) >> 1) * ss + (uint32_t)(W::RAW_ROW + 4 * (lane & 1));
    auto issue = [&](uint8_t* raw) __attribute__((always_inline)) {
      const __amdgpu_buffer_rsrc_t w = __builtin_amdgcn_make_buffer_rsrc(
          const_cast<uint8_t*>(cache_head + (uint64_t)(uint32_t)block * (uint32_t)io.g.stride_block), 0, 0x7fffffff, 0x00020000);
      W::load_half(w, offset, g_chunk, g_tail, raw + (16 * half + first_row) * W::RAW_ROW, raw + W::RAW_TAIL + 256 * half);
    };
    uint8_t* const raws = lds;
    uint8_t* const bufs = lds + 2 * W::RAW_BYTES;
    const typename W::Places places = W::places(tid);
    next_place();
    issue(raws);
    next_place();
    issue(raws + W::RAW_BYTES);
    next_place();

    half8_t qop[KS];
    const int64_t elem = col.row * io.q_stride_t + (int64_t)(col.valid ? col.head : hkv * io.group) * io.q_stride_h;
    if (q_dtype == KVQ_BF16) W::template load_q<KVQ_BF16>(io, elem, col.valid, lane, qop);
    else if (q_dtype == KVQ_F16) W::template load_q<KVQ_F16>(io, elem, col.valid, lane, qop);
    else W::template load_q<KVQ_F32>(io, elem, col.valid, lane, qop);
    const float k_mul = io.scale_log2 * DTile::kKScaleMul;
    float ali = 0.f;
    bool biased = false;
    if constexpr (EXT) {
      biased = io.alibi != nullptr;
      ali = alibi_slope(io.alibi, col.valid ? col.head : hkv * io.group);
    }

    auto fence = []() __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); };
    // every load into LDS of this wave has landed, every LDS access is done, and so for the other waves
    auto tile_barrier = []() __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    tile_barrier();
    typename W::Expand e;
    W::expand_load(e, places, raws);
#pragma unroll
    for (int i = 0; i < 4; ++i) W::expand_k_piece(e, places, i, bufs);
#pragma unroll
    for (int i = 0; i < 5; ++i) W::template expand_v_piece<true>(e, places, i, bufs);
    if (wave == 0) W::expand_scales(e.sc, bufs, k_mul);
    tile_barrier();
    issue(raws);
    next_place();

    const uint32_t op_read = (uint32_t)((lane & 31) * 16 + (lane >> 5) * 512);          // K operand of k-step 0
    const uint32_t v_read = (uint32_t)((lane & 31) * 16 + (lane >> 5) * (D * 16));       // V operand of row tile 0, half 0
    const uint32_t sc_read = (uint32_t)(W::K_BYTES + W::V_BYTES + 4 * (((lane & 15) >> 2) * 8 + 4 * (lane >> 5) + (lane & 3)));
    half8_t ka[KS], va[MT][2];
    float ksc, vsc, allow;
    auto read_k = [&](const uint8_t* buf, int ks) __attribute__((always_inline)) { ka[ks] = *reinterpret_cast<const half8_t*>(buf + op_read + 1024 * ks); };
    auto read_v = [&](const uint8_t* buf, int mt, int kt) __attribute__((always_inline)) {
      va[mt][kt] = *reinterpret_cast<const half8_t*>(buf + W::K_BYTES + v_read + 2 * kt * D * 16 + mt * 512);
    };
    auto tile_begin = [&](const uint8_t* buf, const uint8_t* raw_next) __attribute__((always_inline)) {
#pragma unroll
      for (int ks = 0; ks < KS / 2; ++ks) read_k(buf, ks);
      W::expand_load(e, places, raw_next);
      ksc = *reinterpret_cast<const float*>(buf + sc_read);
      vsc = *reinterpret_cast<const float*>(buf + sc_read + 128);
      allow = *reinterpret_cast<const float*>(buf + W::K_BYTES + W::V_BYTES + 256);
    };
    tile_begin(bufs, raws + W::RAW_BYTES);

    // Step t: products and softmax of tile t; tile t + 1 is expanded, tile t + 3 requested.
    auto step_fn = [&](auto masked, auto parity, int t) __attribute__((always_inline)) {
      constexpr bool MASK = decltype(masked)::value;
      constexpr int P = decltype(parity)::value;
      const uint8_t* buf = bufs + P * W::BUF_BYTES;
      uint8_t* nbuf = bufs + (1 - P) * W::BUF_BYTES;
      u32x4 pb[2];
      floatx16 s;
      // From here to the end of the tile's products the wave outranks the waves of its SIMD that wait or fetch.
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        s = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka[ks], qop[ks], ks == 0 ? (floatx16){} : s, 0, 0, 0);
        if (ks < KS / 2) read_k(buf, KS / 2 + ks);
        if (ks > 0)
#pragma unroll
          for (int j = (ks - 1) * 9 / (KS - 1); j < ks * 9 / (KS - 1); ++j) {
            if (j < 4) W::expand_k_piece(e, places, j, nbuf);
            else W::template expand_v_piece<MASK>(e, places, j - 4, nbuf);
          }
        fence();
      }
      const float d = W::template logits<MASK, EXT>(ksc, io, ali, limit, wspan, t, step_lane, biased, s);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) read_v(buf, mt, 0);
      // The reference maximum only has to keep 2^(logit - m) in range: it stays put while no logit exceeds it by more
      // than the tile's allowance (with 32 columns per wave SOME true maximum moves in most tiles of the first thousand
      // tokens, and each move rescales every accumulator).
      const float thr = seen ? m + allow : -INFINITY;
      if (__builtin_amdgcn_ballot_w64(d > thr) != 0) {
        const float dd = max_over_halves(d);
        const float m_new = dd > thr ? dd : m;   // (a column's reference depends on its own logits only)
        const float alpha = seen ? __builtin_amdgcn_exp2f(m - m_new) : 0.f;
        seen = seen || dd != -INFINITY;
        m = m_new;
        l *= alpha;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) o[mt] *= alpha;
      }
      if (wave == 0) W::expand_scales(e.sc, nbuf, k_mul);
      auto weights = [&](int i) __attribute__((always_inline)) {
        float x[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const float p = __builtin_amdgcn_exp2f(s[2 * i + r] - m);
          l += p;
          x[r] = p * W::row_lane(vsc, 2 * i + r);
        }
        uint32_t w = pack_half2(x[0], x[1]);
        asm volatile("" : "+v"(w), "+v"(l));   // computed here, not where it is used
        pb[i / 4][i % 4] = w;
      };
      auto pv = [&](int mt, int kt) __attribute__((always_inline)) {
        o[mt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[mt][kt], __builtin_bit_cast(half8_t, pb[kt]), o[mt], 0, 0, 0);
      };
#pragma unroll
      for (int i = 0; i < 4; ++i) weights(i);
      fence();
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (i < MT) {
          pv(i, 0);
          read_v(buf, i, 1);
        }
        weights(4 + i);
        fence();
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        pv(mt, 1);
        fence();
      }
      __builtin_amdgcn_s_setprio(0);
      tile_barrier();   // tile t is read, tile t + 1 expanded, tile t + 2 in LDS
      issue(raws + (1 - P) * W::RAW_BYTES);
      next_place();
      tile_begin(nbuf, raws + P * W::RAW_BYTES);
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    // Tiles below every column's limit need no mask.  They and the masked head and tail are separate loops (every wave
    // runs the same number of steps, hence of barriers, whichever loop a step is in).  Step t expands tile t + 1, whose
    // slots past the end of the sequence may hold anything: of account for the conversion of fp8 codes.
    const int t_plain = min(t_hi, min(wave_min_limit, W::FP8 ? len - kTile : len) / kTile) & ~1;
    int t = t_lo;
    if constexpr (EXT) {
      // tiles that straddle a column's lower window edge, and those that hold a slot below every column's (wg_first: also
      // for a wave without a valid column, which expands its share of them like any other)
      const int t_head = min(t_hi, ((max(wave_max_first, wg_first) + kTile - 1) / kTile + 1) & ~1);
      for (; t < t_head; t += 2) {
        step_fn(std::true_type{}, I0{}, t);
        if (t + 1 < t_hi) step_fn(std::true_type{}, I1{}, t + 1);
      }
    }
    for (; t < t_plain; t += 2) {
      step_fn(std::false_type{}, I0{}, t);
      step_fn(std::false_type{}, I1{}, t + 1);
    }
    if (t < t_hi) {   // what the plain steps did not need
      step_lane = (int)W::lane_anew();
      limit = limit_of(column(step_lane));
    }
    for (; t < t_hi; t += 2) {   // (the same end for all waves, in whichever loops they have been)
      step_fn(std::true_type{}, I0{}, t);
      if (t + 1 < t_hi) step_fn(std::true_type{}, I1{}, t + 1);
    }
    // no load may land in LDS after the workgroup has given it up
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }

  const int lane_end = (int)W::lane_anew();
  const Column end = column(lane_end);
  l += __shfl_xor(l, 32, kWave);
  if (!end.valid) return;
  const int g = lane_end >> 5;
  if (nsplit > 1) {
    // the range's state: the row as accumulated (without the factor the weights carry), the reference maximum, the sum
    float* p = a.part + ((end.row * io.num_q_heads + end.head) * nsplit + split) * (D + 2);
    const float unit = 1.0f / DTile::kOutDiv;
#pragma unroll
    for (int i = 0; i < D / 8; ++i) {
      floatx4 v;
#pragma unroll
      for (int b = 0; b < 4; ++b) v[b] = W::o_dim(o, i, b) * unit;
      *reinterpret_cast<floatx4_a4*>(p + W::first_dim(i, g)) = v;
    }
    if (g == 0) {
      p[D] = l > 0.f ? m : -INFINITY;
      p[D + 1] = l;
    }
    return;
  }
  if (l > 0.f) l += sink_term(io.sinks, end.head, m);   // a row without a visible key keeps its zeros
  const float mul = l > 0.f ? 1.0f / (l * DTile::kOutDiv) : 0.f;
  const int64_t base = end.row * io.out_stride_t + (int64_t)end.head * io.out_stride_h;
  // One straight run of stores per output type: a short prompt's launch fetches all of this for the first time (asked for
  // the type and branching on NaN element by element it was 2300 instructions: 70 tokens, 8 kv heads of 128, captured, a step
  // 15.9 us in the kernel that knew its type at compile time, 17.6 so, 15.2 now).
  auto store_row = [&](auto type) __attribute__((always_inline)) {
    constexpr int ODT = decltype(type)::value;
#pragma unroll
    for (int i = 0; i < D / 8; ++i) {
      floatx4 v;
#pragma unroll
      for (int b = 0; b < 4; ++b) v[b] = W::o_dim(o, i, b) * mul;
      const int64_t at = base + W::first_dim(i, g);
      if constexpr (ODT == KVQ_F32) *reinterpret_cast<floatx4_a4*>(reinterpret_cast<float*>(io.out) + at) = v;
      else *reinterpret_cast<u32x2_a4*>(reinterpret_cast<uint16_t*>(io.out) + at) =
          ODT == KVQ_BF16 ? (u32x2){W::pack_bf16(v.x, v.y), W::pack_bf16(v.z, v.w)} : (u32x2){pack_half2(v.x, v.y), pack_half2(v.z, v.w)};
    }
  };
  if (out_dtype == KVQ_BF16) store_row(std::integral_constant<int, KVQ_BF16>{});
  else if (out_dtype == KVQ_F16) store_row(std::integral_constant<int, KVQ_F16>{});
  else store_row(std::integral_constant<int, KVQ_F32>{});
  if (io.lse != nullptr && g == 0)
    io.lse[end.row * io.num_q_heads + end.head] = l > 0.f ? (m + __builtin_amdgcn_logf(l)) * kLn2 : -INFINITY;
}

// The merge of the context splits: grid (query rows, ceil(Hq / 4)), a wave per (row of a run, q head), a lane D / 64 dims.
// The rows are counted over the runs (over every sequence of a mixed batch, most of the blocks would find a decode row:
// 153 us of 330 beside 91 of them): a few sequences by a lane each, more over the plan's, a handful where a launch is split.
// out = sum_s w_s o_s / sum_s w_s l_s with w_s = 2^(m_s - max m): the algebra of
// merge_attn_states over the splits' states; the sink's term and the row's lse as in the unsplit kernel.
// A stream of the states, 520 bytes per split at D = 128: every load of a row leaves before the first is used (splits past
// the last reread it and weigh 0).  One block per row whose four waves went through the heads, and a head's splits, one
// after the other took 26 us for 512 rows x 32 heads x 4 splits (34 MB), this takes 9.
template <int D>
__global__ __launch_bounds__(256) void prefill_split_merge_kernel(PrefillArgs a, int out_dtype) {
  constexpr int V = D / 64;
  typedef float vec_t __attribute__((ext_vector_type(V), aligned(4 * V)));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int head = blockIdx.y * 4 + wave;
  const AttnIO& io = a.io;
  if (head >= io.num_q_heads) return;
  int qi = blockIdx.x;
  int64_t row = -1;
  if (a.plan == nullptr) {
    const int i = min(lane, a.num_seqs - 1);   // (kRunsInKernel of them at most)
    const int q_begin = a.cu_seqlens_q[i], q_len = a.cu_seqlens_q[i + 1] - q_begin;
    const int n = lane < a.num_seqs && q_len > 1 && a.seq_lens[i] > 0 ? q_len : 0;
    const int end = wave_incl_scan(n);
    const uint64_t hit = __builtin_amdgcn_ballot_w64(qi < end && qi >= end - n);
    if (hit == 0) return;
    row = __builtin_amdgcn_readlane(q_begin + qi - (end - n), __builtin_ctzll(hit));
  } else {
    for (int i = 0; i < a.plan[0]; ++i) {   // uniform: scalar loads
      const int seq = a.plan[1 + i];
      const int q_begin = a.cu_seqlens_q[seq], q_len = a.cu_seqlens_q[seq + 1] - q_begin;
      if (qi < q_len) {
        row = q_begin + qi;
        break;
      }
      qi -= q_len;
    }
  }
  if (row < 0) return;
  const int S = a.ksplit;
  const float* p = a.part + ((row * io.num_q_heads + head) * S) * (D + 2);
  const int mine = min(lane, S - 1);   // lane s takes split s's (m, l)
  const float ms = p[mine * (D + 2) + D], ls = p[mine * (D + 2) + D + 1];
  float po[kMaxKSplit][V];
#pragma unroll
  for (int s = 0; s < kMaxKSplit; ++s) {
    const vec_t x = *reinterpret_cast<const vec_t*>(p + min(s, S - 1) * (D + 2) + V * lane);
#pragma unroll
    for (int i = 0; i < V; ++i) po[s][i] = x[i];
  }
  const float mmax = wave_max(ms);
  const float mref = mmax == -INFINITY ? 0.f : mmax;
  const float es = lane < S ? __builtin_amdgcn_exp2f(ms - mref) : 0.f;   // an empty range: 2^-inf = 0
  float l = wave_sum(es != 0.f ? es * ls : 0.f);
  float acc[V];
#pragma unroll
  for (int i = 0; i < V; ++i) acc[i] = 0.f;
#pragma unroll
  for (int s = 0; s < kMaxKSplit; ++s) {
    const float w = as_f32(__builtin_amdgcn_readlane(as_u32(es), s));
    const uint32_t keep = w != 0.f ? 0xffffffffu : 0u;   // a weight of 0 takes the words out, whatever they hold
#pragma unroll
    for (int i = 0; i < V; ++i) acc[i] += w * as_f32(as_u32(po[s][i]) & keep);
  }
  if (l > 0.f) l += sink_term(io.sinks, head, mmax);   // a row without a visible key keeps its zeros
  const float mul = l > 0.f ? 1.0f / l : 0.f;
  const int64_t at = row * io.out_stride_t + (int64_t)head * io.out_stride_h + V * lane;
#pragma unroll
  for (int i = 0; i < V; ++i) store_act_rt(out_dtype, io.out, at + i, acc[i] * mul);
  if (io.lse != nullptr && lane == 0)
    io.lse[row * io.num_q_heads + head] = l > 0.f ? (mmax + __builtin_amdgcn_logf(l)) * kLn2 : -INFINITY;
}

template <int D, bool EXT, int CODE>
static int launch_shared_code(PrefillArgs& a, int max_query_len, int q_dtype, int out_dtype, hipStream_t s) {
  using W = SharedTile<D, CODE>;
  a.q_tokens = W::COLS / a.io.group;
  const int blocks = (max_query_len + a.q_tokens - 1) / a.q_tokens;
  if (a.num_seqs > 65535 || a.io.g.num_kv_heads > 65535) return fail(KVQ_EINVAL, "paged_attn_int8: prefill grid out of range");
  if (a.ksplit < 1) a.ksplit = 1;
  dim3 grid(blocks * a.ksplit, a.num_seqs, a.io.g.num_kv_heads);
  if (a.plan != nullptr)
    hipLaunchKernelGGL((paged_prefill_shared_kernel<D, EXT, CODE, true>), grid, dim3(256), 0, s, a, q_dtype, out_dtype);
  else
    hipLaunchKernelGGL((paged_prefill_shared_kernel<D, EXT, CODE, false>), grid, dim3(256), 0, s, a, q_dtype, out_dtype);
  if (int e = check_hip(hipGetLastError(), "paged_prefill_shared launch")) return e;
  if (a.ksplit == 1) return KVQ_OK;
  dim3 mgrid(a.num_tokens, (a.io.num_q_heads + 3) / 4);
  hipLaunchKernelGGL((prefill_split_merge_kernel<D>), mgrid, dim3(256), 0, s, a, out_dtype);
  return check_hip(hipGetLastError(), "prefill split merge launch");
}

template <int D>
int launch_prefill_shared(PrefillArgs& a, int max_query_len, int q_dtype, int out_dtype, hipStream_t s) {
  const bool ext = a.io.window > 0 || a.io.cap_c != 0.f || a.io.alibi != nullptr;
  switch (a.io.g.code_type) {
    case KVQ_CODE_FP8_E4M3:
      return ext ? launch_shared_code<D, true, KVQ_CODE_FP8_E4M3>(a, max_query_len, q_dtype, out_dtype, s)
                 : launch_shared_code<D, false, KVQ_CODE_FP8_E4M3>(a, max_query_len, q_dtype, out_dtype, s);
    case KVQ_CODE_INT4:
      return ext ? launch_shared_code<D, true, KVQ_CODE_INT4>(a, max_query_len, q_dtype, out_dtype, s)
                 : launch_shared_code<D, false, KVQ_CODE_INT4>(a, max_query_len, q_dtype, out_dtype, s);
    default:
      return ext ? launch_shared_code<D, true, KVQ_CODE_INT8>(a, max_query_len, q_dtype, out_dtype, s)
                 : launch_shared_code<D, false, KVQ_CODE_INT8>(a, max_query_len, q_dtype, out_dtype, s);
  }
}

}  // namespace kvq
