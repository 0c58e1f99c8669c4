// kern_cohort_parts.hip -- the cohort kernels of parts of an iteration (see kernels.hpp).
#include "pipe_kernel.hpp"
#include "kernels.hpp"

namespace brr {
BRR_COHORT_KERNELS(BRR_COHORT_INST, true)
} // namespace brr
