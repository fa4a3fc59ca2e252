// Instantiations of the pipelined window passes, complex128.
#include "fiber_pipe.hpp"

namespace ffsim_amd {
const void* pipe_kernel_c128(int units, int variant) { return pipe_kernel<double>(units, variant); }
}  // namespace ffsim_amd
