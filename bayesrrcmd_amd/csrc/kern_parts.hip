// kern_parts.hip -- the pipelined BayesR sweep kernels of parts of an iteration (see kernels.hpp).
#include "pipe_kernel.hpp"
#include "kernels.hpp"

namespace brr {
BRR_PIPE_KERNELS_OF(BRR_PIPE_INST, false, true)
BRR_PIPE_KERNELS_OF(BRR_PIPE_INST, true, true)
} // namespace brr
