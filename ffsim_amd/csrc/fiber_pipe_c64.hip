// Instantiations of the pipelined window passes, complex64.
#include "fiber_pipe.hpp"

namespace ffsim_amd {
const void* pipe_kernel_c64(int units, int sweeps, int cols, int variant) {
  return pipe_kernel<float>(units, sweeps, cols, variant);
}
}  // namespace ffsim_amd
