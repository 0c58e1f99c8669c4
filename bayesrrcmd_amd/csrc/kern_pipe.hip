// kern_pipe.hip -- the pipelined BayesR sweep kernels with an FP64 residual (see kernels.hpp).
#include "pipe_kernel.hpp"
#include "kernels.hpp"

namespace brr {
BRR_PIPE_KERNELS_OF(BRR_PIPE_INST, false, false)
} // namespace brr
