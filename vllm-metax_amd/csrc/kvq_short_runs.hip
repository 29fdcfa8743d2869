// Host side of the short-run launch.
#include "kvq_short_runs_impl.cuh"

namespace kvq {

extern template int launch_short_runs_d<64>(const ShortRunArgs& args, hipStream_t s);
extern template int launch_short_runs_d<128>(const ShortRunArgs& args, hipStream_t s);

static size_t state_rows(const ShortRunArgs& a, int num_kv_heads) {
  return 2 * (size_t)a.num_wg * (size_t)num_kv_heads * (size_t)a.rows;
}

bool short_runs_shape(int num_q_heads, int num_kv_heads, int head_size, int num_seqs, int max_query_len, int num_wg,
                      ShortRunArgs* a, size_t* bytes) {
  const int group = num_q_heads / num_kv_heads;
  if (max_query_len < 2 || (int64_t)max_query_len * group > kShortRunCols || batch_invariant()) return false;
  if (head_size > 128) return false;   // two windows per wave would not fit the LDS, a tile in registers spills
  a->cols = max_query_len * group > 16 ? 32 : 16;
  a->q_tokens = max_query_len < a->cols / group ? max_query_len : a->cols / group;
  a->rows = a->q_tokens * group;
  a->blocks = (max_query_len + a->q_tokens - 1) / a->q_tokens;
  a->num_seqs = num_seqs;
  a->num_wg = num_wg;
  *bytes = state_rows(*a, num_kv_heads) * (head_size + 2) * sizeof(float) + (1 + (size_t)num_seqs * a->blocks) * sizeof(int64_t);
  return (int64_t)num_seqs * a->blocks <= 0x7fffffff / 64 && state_rows(*a, num_kv_heads) <= 0x7fffffff;
}

bool short_runs_cache(const kvq_cache_geom& g) { return g.stride_slot == 2 * (code_bytes(g) + 4); }

int launch_short_runs(ShortRunArgs& a, void* workspace, int out_dtype, hipStream_t s) {
  if (out_dtype != KVQ_F32 && out_dtype != KVQ_BF16 && out_dtype != KVQ_F16)
    return fail(KVQ_EINVAL, "paged_attn_int8: unknown out_dtype %d", out_dtype);
  if (a.q_dtype != KVQ_F32 && a.q_dtype != KVQ_BF16 && a.q_dtype != KVQ_F16)
    return fail(KVQ_EINVAL, "paged_attn_int8: unknown q_dtype %d", a.q_dtype);
  const size_t rows = state_rows(a, a.io.g.num_kv_heads);
  a.part_o = static_cast<float*>(workspace);
  a.part_ml = a.part_o + rows * a.io.g.head_size;
  a.line = reinterpret_cast<int64_t*>(a.part_ml + 2 * rows);
  switch (a.io.g.head_size) {
    case 64: return launch_short_runs_d<64>(a, s);
    default: return launch_short_runs_d<128>(a, s);
  }
}

}  // namespace kvq

extern "C" size_t kvq_paged_attn_short_runs_workspace_bytes(int max_num_seqs, int num_q_heads, int num_kv_heads,
                                                            int head_size, int max_query_len) {
  using namespace kvq;
  if (max_num_seqs <= 0 || num_kv_heads <= 0 || num_q_heads < num_kv_heads || num_q_heads % num_kv_heads != 0 ||
      (head_size != 64 && head_size != 128) || num_q_heads / num_kv_heads > 16)
    return 0;
  const int longest = kShortRunCols / (num_q_heads / num_kv_heads);
  ShortRunArgs a{};
  size_t bytes = 0;
  if (!short_runs_shape(num_q_heads, num_kv_heads, head_size, max_num_seqs, max_query_len == 0 ? longest : max_query_len,
                        num_cus(), &a, &bytes))
    return 0;
  const size_t plain = kvq_paged_attn_workspace_bytes(max_num_seqs, num_q_heads, head_size);
  return bytes > plain ? bytes : plain;
}
