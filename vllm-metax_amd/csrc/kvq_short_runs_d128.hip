// Short-run kernels for head size 128.
#include "kvq_short_runs_impl.cuh"

namespace kvq {
template int launch_short_runs_d<128>(const ShortRunArgs& args, hipStream_t s);
}  // namespace kvq
