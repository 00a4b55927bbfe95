// Fused drop kernels of 2x2 links for heterogeneous classes with the alternative FFT values per thread.
#include "hpx_drop.hpp"

namespace hpx {

int batch_launch_alt_2(const void* plans_dev, const hpx_uneven_class& c, hipStream_t s) {
  return launch_multi<2, true>(static_cast<const BatchArgs*>(plans_dev), c, s);
}

}  // namespace hpx
