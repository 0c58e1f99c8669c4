// kern_gram.hip -- the Gram entries of a sweep's blocks (see kernels.hpp).
#include "gram_kernel.hpp"
#include "kernels.hpp"

namespace brr {
BRR_GRAM_INST(false)
BRR_GRAM_INST(true)
} // namespace brr
