// Chunked prefill over the paged cache: the plan of a launch and the dispatch by head size.
#include "kvq_prefill_impl.cuh"

namespace kvq {

extern template int launch_prefill_q<64>(PrefillArgs& a, int max_query_len, int q_dtype, int out_dtype, hipStream_t s);
extern template int launch_prefill_q<128>(PrefillArgs& a, int max_query_len, int q_dtype, int out_dtype, hipStream_t s);
extern template int launch_prefill_q<256>(PrefillArgs& a, int max_query_len, int q_dtype, int out_dtype, hipStream_t s);

// The plan where no decode launch ahead of this one has written it (write_prefill_plan).
__global__ __launch_bounds__(64) void prefill_plan_kernel(const int32_t* seq_lens, const int32_t* cu_seqlens_q,
                                                          int num_seqs, int32_t* plan) {
  write_prefill_plan(seq_lens, cu_seqlens_q, num_seqs, plan);
}

bool prefill_needs_plan(int num_seqs, int head_size, int max_query_len, int group) {
  return num_seqs > kRunsInKernel || batch_invariant() || !takes_shared_tile(head_size, max_query_len, group);
}

int launch_prefill(const AttnIO& io, const int32_t* seq_lens, const int32_t* cu_seqlens_q, int num_seqs,
                   int max_query_len, int causal, int q_dtype, int out_dtype, int32_t* plan, bool planned,
                   hipStream_t s, int ksplit, int num_tokens, float* part) {
  PrefillArgs a{};
  a.ksplit = ksplit;
  a.num_tokens = num_tokens;
  a.part = part;
  a.io = io;
  a.seq_lens = seq_lens;
  a.cu_seqlens_q = cu_seqlens_q;
  a.num_seqs = num_seqs;
  a.causal = causal;
  if (prefill_needs_plan(num_seqs, io.g.head_size, max_query_len, io.group)) {
    a.plan = plan;
    if (!planned) {
      hipLaunchKernelGGL(prefill_plan_kernel, dim3(1), dim3(64), 0, s, seq_lens, cu_seqlens_q, num_seqs, plan);
      if (int e = check_hip(hipGetLastError(), "prefill plan launch")) return e;
    }
  }
  switch (io.g.head_size) {
    case 64: return launch_prefill_q<64>(a, max_query_len, q_dtype, out_dtype, s);
    case 128: return launch_prefill_q<128>(a, max_query_len, q_dtype, out_dtype, s);
    default: return launch_prefill_q<256>(a, max_query_len, q_dtype, out_dtype, s);
  }
}

}  // namespace kvq
