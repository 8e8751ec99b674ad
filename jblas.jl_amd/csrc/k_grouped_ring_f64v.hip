// k_grouped_ring_f64v.hip -- grouped FP64 kernels with 16-byte operand loads.
#include "k_grouped_ring.h"

namespace jb {
GroupedKernelFn grouped_ring_f64_vec(int which, int combo) { return ring_kernel_of<double, true>(which, combo); }
}  // namespace jb
