// kern_sweep_seq.hip -- the round-by-round BayesR sweep kernels (see kernels.hpp).
#include "sweep_kernel.hpp"
#include "kernels.hpp"

namespace brr {
BRR_SWEEP_SEQ_KERNELS(BRR_SWEEP_INST)
} // namespace brr
