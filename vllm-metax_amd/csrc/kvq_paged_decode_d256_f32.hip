// Paged decode kernels for head size 256, fp32 queries.
#include "kvq_paged_decode_impl.cuh"

namespace kvq {
template int launch_streamk<256, KVQ_F32>(const StreamKArgs& args, hipStream_t s);
template int launch_v2<256, KVQ_F32>(const V2Args& a, int num_seqs, hipStream_t s);
}  // namespace kvq
