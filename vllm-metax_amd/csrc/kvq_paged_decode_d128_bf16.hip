// Paged decode kernels for head size 128, bf16 queries.
#include "kvq_paged_decode_impl.cuh"

namespace kvq {
template int launch_streamk<128, KVQ_BF16>(const StreamKArgs& args, hipStream_t s);
template int launch_v2<128, KVQ_BF16>(const V2Args& a, int num_seqs, hipStream_t s);
}  // namespace kvq
