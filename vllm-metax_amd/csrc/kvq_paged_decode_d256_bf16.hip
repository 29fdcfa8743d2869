// Paged decode kernels for head size 256, bf16 queries.
#include "kvq_paged_decode_impl.cuh"

namespace kvq {
template int launch_streamk<256, KVQ_BF16>(const StreamKArgs& args, hipStream_t s);
template int launch_v2<256, KVQ_BF16>(const V2Args& a, int num_seqs, hipStream_t s);
}  // namespace kvq
