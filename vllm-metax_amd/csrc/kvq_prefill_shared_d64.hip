// The workgroup-shared prefill tile for head size 64.
#include "kvq_prefill_shared.cuh"

namespace kvq {
template int launch_prefill_shared<64>(PrefillArgs& a, int max_query_len, int q_dtype, int out_dtype, hipStream_t s);
}  // namespace kvq
