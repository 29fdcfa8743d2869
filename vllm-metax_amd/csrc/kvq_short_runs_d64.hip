// Short-run kernels for head size 64.
#include "kvq_short_runs_impl.cuh"

namespace kvq {
template int launch_short_runs_d<64>(const ShortRunArgs& args, hipStream_t s);
}  // namespace kvq
