// kern_pipe_f32.hip -- the pipelined BayesR sweep kernels with an FP32 residual and FP64 refresh (see
// kernels.hpp).
#include "pipe_kernel.hpp"
#include "kernels.hpp"

namespace brr {
BRR_PIPE_KERNELS_OF(BRR_PIPE_INST, true, false)
} // namespace brr
