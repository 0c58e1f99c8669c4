// kern_sweep_async.hip -- the BayesR sweep kernels in asynchronous windows (see kernels.hpp).
#include "sweep_kernel.hpp"
#include "kernels.hpp"

namespace brr {
BRR_SWEEP_ASYNC_KERNELS(BRR_SWEEP_INST)
} // namespace brr
