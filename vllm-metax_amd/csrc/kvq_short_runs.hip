// Host side of the short-run launch.
#include "kvq_short_runs_impl.cuh"

namespace kvq {

extern template int launch_short_runs_d<64>(const ShortRunArgs& args, hipStream_t s);
extern template int launch_short_runs_d<128>(const ShortRunArgs& args, hipStream_t s);

bool short_runs_take(const kvq_cache_geom& g, int num_q_heads, int num_seqs, int max_query_len, int num_wg, ShortRunArgs* a,
                     size_t* bytes) {
  const int group = num_q_heads / g.num_kv_heads;
  if (max_query_len < 2 || (int64_t)max_query_len * group > kShortRunCols || batch_invariant()) return false;
  if (g.stride_slot != 2 * (code_bytes(g) + 4)) return false;   // records of a head back to back
  if (g.head_size > 128) return false;   // two windows per wave would not fit the LDS, a tile in registers spills
  a->cols = max_query_len * group > 16 ? 32 : 16;
  a->q_tokens = a->cols / group;
  a->blocks = (max_query_len + a->q_tokens - 1) / a->q_tokens;
  a->num_seqs = num_seqs;
  a->num_wg = num_wg;
  const size_t rows = ((size_t)num_wg + (size_t)num_seqs * a->blocks) * g.num_kv_heads * a->cols;
  *bytes = rows * (g.head_size + 2) * sizeof(float) + (1 + (size_t)num_seqs * a->blocks) * sizeof(int64_t);
  return (int64_t)num_seqs * a->blocks <= 0x7fffffff / 64;
}

int launch_short_runs(ShortRunArgs& a, void* workspace, int out_dtype, hipStream_t s) {
  if (out_dtype != KVQ_F32 && out_dtype != KVQ_BF16 && out_dtype != KVQ_F16)
    return fail(KVQ_EINVAL, "paged_attn_int8: unknown out_dtype %d", out_dtype);
  if (a.q_dtype != KVQ_F32 && a.q_dtype != KVQ_BF16 && a.q_dtype != KVQ_F16)
    return fail(KVQ_EINVAL, "paged_attn_int8: unknown q_dtype %d", a.q_dtype);
  const size_t rows = ((size_t)a.num_wg + (size_t)a.num_seqs * a.blocks) * a.io.g.num_kv_heads * a.cols;
  a.part_o = static_cast<float*>(workspace);
  a.part_ml = a.part_o + rows * a.io.g.head_size;
  a.line = reinterpret_cast<int64_t*>(a.part_ml + 2 * rows);
  switch (a.io.g.head_size) {
    case 64: return launch_short_runs_d<64>(a, s);
    default: return launch_short_runs_d<128>(a, s);
  }
}

}  // namespace kvq
