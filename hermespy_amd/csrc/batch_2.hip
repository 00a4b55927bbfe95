// Fused drop kernels of 2x2 links: single-link launches, and heterogeneous classes with the default FFT
// values per thread.
#include "hpx_drop.hpp"

namespace hpx {

int batch_launch_single_2(const void* plan, int64_t num_drops, hipStream_t s) {
  return launch_single<2>(*static_cast<const Plan*>(plan), num_drops, s);
}

int batch_launch_multi_2(const void* plans_dev, const hpx_uneven_class& c, hipStream_t s) {
  return launch_multi<2, false>(static_cast<const BatchArgs*>(plans_dev), c, s);
}

}  // namespace hpx
