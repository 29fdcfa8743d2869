// Prefill kernels for head size 128.
#include "kvq_prefill_impl.cuh"

namespace kvq {
template int launch_prefill_q<128>(PrefillArgs& a, int max_query_len, int q_dtype, int out_dtype, hipStream_t s);
}  // namespace kvq
