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
// columns are at least half full).  One short run takes the whole batch with it, also where it is alone among decode rows,
// which then compute 16 or 32 columns each.  Measured on MI355X against the decode and prefill kernels on 308 batches
// (0 .. 200 decode rows, 1 .. 64 runs of up to 3 or 8 tokens, 100 - 2000 or 1k - 8k tokens each, 4 to 32 kv heads and one):
//   16 columns: 1.07 .. 1.5 times as fast in the mean at every batch size; slower where 16 runs stand alone on 16 or 32 kv
//     heads (61.0 against 46.9 us at worst);
//   32 columns: 1.4 .. 2.5 times up to 40 sequences, 1.1 .. 1.6 up to 180, beyond that 1.0 on short contexts (0.87 .. 1.18)
//     and 1.15 on long ones;
//   one run beside 8 / 32 / 64 / 128 / 200 decode rows: 1.6 / 1.3 / 1.3 / 1.15 / 1.08 in the median, 0.91 at worst.
// No line between the batches that lose and those that gain follows from what the host knows of a launch.
constexpr int kShortRunCols = 63;

// Whether the launch can serve a batch of these sizes, the shape of its items, and the bytes of 16-byte aligned workspace
// it needs: more sequences or longer runs never need fewer.
bool short_runs_shape(int num_q_heads, int num_kv_heads, int head_size, int num_seqs, int max_query_len, int num_wg,
                      ShortRunArgs* a, size_t* bytes);
// ... and this cache: head-major, whose blocks it can stream.
bool short_runs_cache(const kvq_cache_geom& g);
int launch_short_runs(ShortRunArgs& a, void* workspace, int out_dtype, hipStream_t s);

}  // namespace kvq
