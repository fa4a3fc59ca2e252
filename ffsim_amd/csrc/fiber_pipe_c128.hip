// Instantiations of the pipelined window passes, complex128.
#include "fiber_pipe.hpp"

namespace ffsim_amd {
const void* pipe_kernel_c128(int units, int sweeps, int cols, int variant) {
  return pipe_kernel<double>(units, sweeps, cols, variant);
}
}  // namespace ffsim_amd
