// k_grouped_ring_f64.hip -- grouped FP64 ring kernels.
#include "k_grouped_ring.h"

namespace jb {
GroupedKernelFn grouped_ring_f64(int which, int combo) { return ring_kernel_of<double>(which, combo); }
GroupedKernelFn grouped_ring_f64_wide_ld(int combo) { return ring_wide_ld_kernel<double>(combo); }
}  // namespace jb
