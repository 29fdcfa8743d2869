// Chunked prefill over the paged cache: the plan of a launch and the dispatch by head size.
#include "kvq_prefill_impl.cuh"

namespace kvq {

extern template int launch_prefill_q<64>(PrefillArgs& a, int max_query_len, int q_dtype, int out_dtype, hipStream_t s);
extern template int launch_prefill_q<128>(PrefillArgs& a, int max_query_len, int q_dtype, int out_dtype, hipStream_t s);
extern template int launch_prefill_q<256>(PrefillArgs& a, int max_query_len, int q_dtype, int out_dtype, hipStream_t s);

// One workgroup lists the sequences that have work for the prefill kernels.  A mixed batch is mostly decode rows;
// a grid over all sequences would spend most of its workgroups finding that out one by one, in between the ones
// that have work.
__global__ __launch_bounds__(64) void prefill_plan_kernel(const int32_t* seq_lens, const int32_t* cu_seqlens_q,
                                                          int num_seqs, int32_t* plan) {
  const int lane = threadIdx.x;
  int count = 0;
  for (int base = 0; base < num_seqs; base += kWave) {
    const int s = base + lane;
    const int sc = s < num_seqs ? s : num_seqs - 1;
    const bool has = s < num_seqs && cu_seqlens_q[sc + 1] - cu_seqlens_q[sc] > 1 && seq_lens[sc] > 0;
    const uint64_t mask = __builtin_amdgcn_ballot_w64(has);
    if (has) plan[1 + count + __builtin_popcountll(mask & ((1ull << lane) - 1))] = s;
    count += __builtin_popcountll(mask);
  }
  if (lane == 0) plan[0] = count;
  // Up to 64 of them are put longest sequence first: their workgroups start in the plan's order, and the
  // longest sequence's are the ones that should not start last.
  if (count > 1 && count <= kWave) {
    __threadfence_block();
    const int id = plan[1 + (lane < count ? lane : 0)];
    const int key = lane < count ? seq_lens[id] : -1;
    int rank = 0;
    for (int j = 0; j < count; ++j) {
      const int kj = __shfl(key, j, kWave);
      rank += (kj > key || (kj == key && j < lane)) ? 1 : 0;
    }
    if (lane < count) plan[1 + rank] = id;
  }
}

int launch_prefill(const AttnIO& io, const int32_t* seq_lens, const int32_t* cu_seqlens_q, int num_seqs,
                   int max_query_len, int causal, int q_dtype, int out_dtype, int32_t* plan, hipStream_t s,
                   int ksplit, int num_tokens, float* part) {
  PrefillArgs a{};
  a.ksplit = ksplit;
  a.num_tokens = num_tokens;
  a.part = part;
  a.io = io;
  a.seq_lens = seq_lens;
  a.cu_seqlens_q = cu_seqlens_q;
  a.num_seqs = num_seqs;
  a.causal = causal;
  a.plan = plan;
  hipLaunchKernelGGL(prefill_plan_kernel, dim3(1), dim3(64), 0, s, seq_lens, cu_seqlens_q, num_seqs, plan);
  if (int e = check_hip(hipGetLastError(), "prefill plan launch")) return e;
  switch (io.g.head_size) {
    case 64: return launch_prefill_q<64>(a, max_query_len, q_dtype, out_dtype, s);
    case 128: return launch_prefill_q<128>(a, max_query_len, q_dtype, out_dtype, s);
    default: return launch_prefill_q<256>(a, max_query_len, q_dtype, out_dtype, s);
  }
}

}  // namespace kvq
