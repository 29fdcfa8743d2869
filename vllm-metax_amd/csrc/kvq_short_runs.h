// Arguments and host entry of the short-run launch (kvq_short_runs_impl.cuh).
#pragma once

#include "kvq_attn_core.cuh"

namespace kvq {

struct ShortRunArgs {
  AttnIO io;
  const int32_t* seq_lens;
  const int32_t* cu_seqlens_q;
  int num_seqs;
  int causal;
  int q_dtype;
  int q_tokens;   // query tokens per item
  int blocks;     // items per sequence: ceil(longest run / q_tokens)
  int cols;       // columns per item, 16 or 32
  int rows;       // of them used: q_tokens x group
  int num_wg;     // P
  int setup_units;
  // Partial states, [Hkv][rows] each.  A workgroup leaves at most two: of the item its share begins inside (slot 2 w) and
  // of the item it ends inside (slot 2 w + 1, which begins with the item's first tile), so their room does not depend on
  // the batch.
  float* part_o;
  float* part_ml;
  int64_t* line;  // [0] the line's length, [1 + i] item i's first unit
};

// Longest run x q heads per kv head up to which a batch's runs are short (beyond it the workgroup-shared tile's 128
// columns are at least half full).
constexpr int kShortRunCols = 63;

// Whether the launch can serve a batch of these sizes, the shape of its items, and the bytes of 16-byte aligned workspace
// it needs: more sequences or longer runs never need fewer.
bool short_runs_shape(int num_q_heads, int num_kv_heads, int head_size, int num_seqs, int max_query_len, int num_wg,
                      ShortRunArgs* a, size_t* bytes);
// ... and this cache: head-major, whose blocks it can stream.
bool short_runs_cache(const kvq_cache_geom& g);
int launch_short_runs(ShortRunArgs& a, void* workspace, int out_dtype, hipStream_t s);

}  // namespace kvq
