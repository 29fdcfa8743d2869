// The per-wave tile of query runs: PrefillTile folds (query token, q head of the group) pairs into the MFMA's columns
// (see kvq_prefill_impl.cuh) and streams a kv head's records with the decode tile's load / stage machinery.
#pragma once

#include "kvq_attn_core.cuh"

namespace kvq {

template <int D, int QDT, int ODT, int NT, int CODE = KVQ_CODE_INT8, bool STREAM = false, bool SCARCE = (NT > 1 && STREAM)>
struct PrefillTile {
  using DTile = DecodeTile<D, QDT, ODT, CODE, STREAM>;
  static constexpr bool FP8 = DTile::FP8;
  static constexpr bool INT4 = DTile::INT4;
  static constexpr int KSTEPS = DTile::KSTEPS;
  static constexpr int DT = DTile::DT;
  static constexpr int VB = DTile::VB;
  static constexpr int PITCH = DTile::PITCH;
  static constexpr int LDS_TILE = DTile::LDS_TILE;
  // SCARCE: two column tiles, or one of head size 256, in an eight-wave workgroup.  The steps are kept in order, since the
  // scheduler would otherwise read and convert operands so far ahead that accumulators spill.
  static constexpr bool kScarce = SCARCE;

  struct State {
    floatx4 o[NT][DT];
    floatx4 psum[NT];
    float m[NT], l[NT];
  };

  // S^T = K . Q^T for NT column tiles, online softmax with a per-column visible-token limit.
  // A column sees tokens [limit - wspan, limit): wspan is the sliding window, or 2^31 - 1 without one.
  // EXT: the logits may pass through the soft cap and take the ALiBi bias (else neither is looked at).
  // (Always inlined: called as a function, as the compiler chose for two column tiles with the extras, it keeps its arrays
  // in scratch memory; 37 runs of 2-7 tokens on windows of 761 took 98.7 us so.)
  template <bool MASK, bool EXT = true>
  __device__ __forceinline__ static void qk_softmax(const AttnIO& io, const LaneOffsets& lo, const half8_t (&qb)[NT][KSTEPS],
                                    const float (&s_init)[NT], const int (&limit)[NT], uint32_t wspan, int t, int lane,
                                    const uint8_t* lds, State& st, half8_t (&p_op)[NT], const float (&ali)[NT]) {
    const int g = lane >> 4;
    const float* sc_lds = reinterpret_cast<const float*>(lds + LDS_TILE);
    floatx4 s[NT][2];
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      s[nt][0] = (floatx4){s_init[nt], s_init[nt], s_init[nt], s_init[nt]};
      s[nt][1] = s[nt][0];
    }
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      if constexpr (INT4) {
        if constexpr (kScarce) DTile::phase_fence();
        half8_t ka[KSTEPS];
        DTile::k_operands_int4(lo, mt, lds, ka);
#pragma unroll
        for (int kk = 0; kk < KSTEPS; ++kk)
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
            s[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ka[kk], qb[nt][kk], s[nt][mt], 0, 0, 0);
      } else {
#pragma unroll
      for (int i = 0; i < KSTEPS / 2; ++i) {
        if constexpr (kScarce) DTile::phase_fence();
        const u32x4 w = DTile::k_chunk(lo, mt, i, lds);
        const half8_t a0 = dequant8<FP8>(w.x, w.y), a1 = dequant8<FP8>(w.z, w.w);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) {
          s[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a0, qb[nt][2 * i], s[nt][mt], 0, 0, 0);
          s[nt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a1, qb[nt][2 * i + 1], s[nt][mt], 0, 0, 0);
        }
      }
      }
    }
    const int tok0 = DTile::s_token(g, 0, 0), tok1 = DTile::s_token(g, 1, 0);
    const floatx4 ks0 = *reinterpret_cast<const floatx4*>(sc_lds + tok0);
    const floatx4 ks1 = *reinterpret_cast<const floatx4*>(sc_lds + tok1);
    const floatx4 vs0 = *reinterpret_cast<const floatx4*>(sc_lds + 32 + tok0);
    const floatx4 vs1 = *reinterpret_cast<const floatx4*>(sc_lds + 32 + tok1);
    const int tok_base = t * kTile + tok0;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      if constexpr (kScarce) DTile::phase_fence();
      float logit[8];
      float mloc = -INFINITY;
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) logit[mt * 4 + i] = s[nt][mt][i] * (mt ? ks1 : ks0)[i];
      }
      if constexpr (EXT) soft_cap(logit, io.cap_c, io.cap_k);
      if (EXT && io.alibi != nullptr) {   // uniform; the column's query stands at limit - 1
        const float rel0 = (float)(tok_base - (limit[nt] - 1));
#pragma unroll
        for (int j = 0; j < 8; ++j) logit[j] = __builtin_fmaf(ali[nt], rel0 + (float)DTile::p_token(j), logit[j]);
      }
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float x = logit[mt * 4 + i];
          if constexpr (MASK) x = ((uint32_t)(limit[nt] - 1 - (tok_base + DTile::p_token(mt * 4 + i))) < wspan) ? x : -INFINITY;
          logit[mt * 4 + i] = x;
          mloc = fmaxf(mloc, x);
        }
      }
      mloc = max_over_quarters(mloc);
      const float m_new = fmaxf(st.m[nt], mloc);
      // a column that has seen no visible token yet keeps m = -inf; exponents are then taken
      // against 0 so that they come out as exp2(-inf) = 0 and never as (-inf) - (-inf)
      const float m_ref = m_new == -INFINITY ? 0.f : m_new;
      if (__builtin_amdgcn_ballot_w64(m_new > st.m[nt]) != 0) {
        const float alpha = __builtin_amdgcn_exp2f(st.m[nt] - m_ref);
        st.l[nt] *= alpha;
        st.psum[nt] *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) st.o[nt][dt] *= alpha;
      }
      st.m[nt] = m_new;
      float pt[8];
#pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int j = mt * 4 + i;
          const float p = __builtin_amdgcn_exp2f(logit[j] - m_ref);
          st.l[nt] += p;
          float x = p * (mt ? vs1 : vs0)[i];
          if constexpr (MASK) x = ((uint32_t)(limit[nt] - 1 - (tok_base + DTile::p_token(mt * 4 + i))) < wspan) ? x : 0.f;
          pt[j] = x;
        }
      }
      u32x4 pb;
      pb.x = pack_half2(pt[0], pt[1]);
      pb.y = pack_half2(pt[2], pt[3]);
      pb.z = pack_half2(pt[4], pt[5]);
      pb.w = pack_half2(pt[6], pt[7]);
      p_op[nt] = __builtin_bit_cast(half8_t, pb);
    }
  }

  // pv() of a tile whose slots do not all hold a token of the window when `garbage` (uniform): those past the sequence's
  // end, and those below the window, whose block the engine may have given back.  Only fp8 bytes need the distinction.
  __device__ __forceinline__ static void pv_any(bool garbage, const LaneOffsets& lo, const half8_t (&p_op)[NT],
                                                const uint8_t* lds, State& st) {
    if (FP8 && garbage) pv<true>(lo, p_op, lds, st);
    else pv<false>(lo, p_op, lds, st);
  }

  // O^T += (V + 1152)^T . P~^T: every converted V operand feeds the NT column tiles.  MASK as in DecodeTile::pv.
  template <bool MASK>
  __device__ __forceinline__ static void pv(const LaneOffsets& lo, const half8_t (&p_op)[NT], const uint8_t* lds, State& st) {
    if constexpr (!FP8) {
      const half_t one = (half_t)1.0f;
      const half8_t ones = {one, one, one, one, one, one, one, one};
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
        st.psum[nt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ones, p_op[nt], st.psum[nt], 0, 0, 0);
    }
    if constexpr (INT4) {
#pragma unroll
      for (int u = 0; u < VB / 2; ++u) {
        if constexpr (kScarce) DTile::phase_fence();
        half8_t va[4];
        DTile::v_operands_int4(lo, u, lds, va);
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
            st.o[nt][4 * u + n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va[n], p_op[nt], st.o[nt][4 * u + n], 0, 0, 0);
      }
      return;
    }
#pragma unroll
    for (int w = 0; w < VB / 4; ++w) {
      if constexpr (kScarce) DTile::phase_fence();
      uint32_t x0[4], x1[4];
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const int ja = 2 * a, jb = 2 * a + 1;
        const uint32_t ta = prep_codes<FP8>(*reinterpret_cast<const uint32_t*>(lds + DTile::v_off(lo, ja, w)));
        const uint32_t tb = prep_codes<FP8>(*reinterpret_cast<const uint32_t*>(lds + DTile::v_off(lo, jb, w)));
        x0[a] = perm(tb, ta, 0x05010400u);
        x1[a] = perm(tb, ta, 0x07030602u);
      }
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        u32x4 av;
        const uint32_t* x = (b < 2) ? x0 : x1;
        av.x = codes_to_half2<FP8, MASK>(x[0], b & 1);
        av.y = codes_to_half2<FP8, MASK>(x[1], b & 1);
        av.z = codes_to_half2<FP8, MASK>(x[2], b & 1);
        av.w = codes_to_half2<FP8, MASK>(x[3], b & 1);
        const half8_t a_op = __builtin_bit_cast(half8_t, av);
        const int dt = 4 * w + b;
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          st.o[nt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a_op, p_op[nt], st.o[nt][dt], 0, 0, 0);
      }
    }
  }

  // ---- several waves on one item: their states meet in LDS, one column tile at a time.  A wave drops the tile's
  //      state into its own window (free once its tiles are done); the item's first wave folds them into its own.
  //      A column may have seen nothing in a wave's tiles (m = -inf): its weight is then 0, never 2^(-inf + inf).
  __device__ static void dump_state(const State& st, int nt, int lane, uint8_t* lds) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<floatx4*>(lds + (dt * 64 + lane) * 16) = st.o[nt][dt];
    *reinterpret_cast<floatx4*>(lds + (DT * 64 + lane) * 16) = (floatx4){st.psum[nt][0], st.m[nt], st.l[nt], 0.f};
  }
  __device__ static void fold_state(State& st, int nt, int lane, const uint8_t* lds) {
    const floatx4 x = *reinterpret_cast<const floatx4*>(lds + (DT * 64 + lane) * 16);
    const float mj = x.y;
    const float m_new = fmaxf(st.m[nt], mj);
    const float m_ref = m_new == -INFINITY ? 0.f : m_new;
    const float a = __builtin_amdgcn_exp2f(st.m[nt] - m_ref);
    const float b = __builtin_amdgcn_exp2f(mj - m_ref);
    st.m[nt] = m_new;
    st.l[nt] = st.l[nt] * a + x.z * b;
    st.psum[nt] = st.psum[nt] * a + x.x * b;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
      st.o[nt][dt] = st.o[nt][dt] * a + *reinterpret_cast<const floatx4*>(lds + (dt * 64 + lane) * 16) * b;
  }

  // The lane's D / 4 dims of column tile `nt` in the order of DTile::out_dim, code bias removed, scaled by `mul`.
  __device__ static void gather_row(const State& st, int nt, float mul, float (&v)[D / 4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        v[DTile::gather_pos(i, dt)] = (st.o[nt][dt][i] - DTile::v_bias(dt) * st.psum[nt][0]) * (mul * DTile::v_unit(dt));
  }
  // The sum of column tile `nt` over the lane's quarters (every lane takes part).
  __device__ static float total_l(const State& st, int nt) {
    float l = st.l[nt];
    l += __shfl_xor(l, 16, kWave);
    l += __shfl_xor(l, 32, kWave);
    return l;
  }

  // Normalise column tile `nt` and write the lane's quarter of its output row.
  __device__ static void emit(const AttnIO& io, int nt, int64_t row, int head, bool valid, int lane, const State& st) {
    if constexpr (ODT == kRuntimeDtype) {
      if (io.out_dtype == KVQ_F32) emit_as<KVQ_F32>(io, nt, row, head, valid, lane, st);
      else if (io.out_dtype == KVQ_BF16) emit_as<KVQ_BF16>(io, nt, row, head, valid, lane, st);
      else emit_as<KVQ_F16>(io, nt, row, head, valid, lane, st);
    } else {
      emit_as<ODT>(io, nt, row, head, valid, lane, st);
    }
  }
  template <int OT>
  __device__ static void emit_as(const AttnIO& io, int nt, int64_t row, int head, bool valid, int lane, const State& st) {
    float l = total_l(st, nt);
    if (!valid) return;
    if (l > 0.f) l += sink_term(io.sinks, head, st.m[nt]);   // a row without a visible key keeps its zeros
    const int g = lane >> 4;
    float v[D / 4];
    gather_row(st, nt, l > 0.f ? 1.0f / (l * DTile::kOutDiv) : 0.f, v);   // no visible key: zeros
    const int64_t base = row * io.out_stride_t + (int64_t)head * io.out_stride_h;
    if constexpr (OT == KVQ_F32) {
      float* o = reinterpret_cast<float*>(io.out) + base;
#pragma unroll
      for (int i = 0; i < D / 4; i += 4) *reinterpret_cast<floatx4_a4*>(o + DTile::out_dim(g, i)) = (floatx4){v[i], v[i + 1], v[i + 2], v[i + 3]};
    } else {
      uint16_t* o = reinterpret_cast<uint16_t*>(io.out) + base;
#pragma unroll
      for (int i = 0; i < D / 4; i += 8) {
        u32x4 pk;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          uint32_t w;
          if constexpr (OT == KVQ_BF16) {
            w = (uint32_t)f32_to_bf16_bits(v[i + 2 * j]) | ((uint32_t)f32_to_bf16_bits(v[i + 2 * j + 1]) << 16);
          } else {
            w = pack_half2(v[i + 2 * j], v[i + 2 * j + 1]);
          }
          pk[j] = w;
        }
        *reinterpret_cast<u32x4_a4*>(o + DTile::out_dim(g, i)) = pk;
      }
    }
    if (io.lse != nullptr && g == 0)
      io.lse[row * io.num_q_heads + head] = l > 0.f ? (st.m[nt] + __builtin_amdgcn_logf(l)) * kLn2 : -INFINITY;
  }
};

}  // namespace kvq
