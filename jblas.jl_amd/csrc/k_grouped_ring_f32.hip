// k_grouped_ring_f32.hip -- grouped native FP32 kernels.
#include "k_grouped_ring.h"

namespace jb {
GroupedKernelFn grouped_ring_f32(int which, int combo) { return ring_kernel_of<float>(which, combo); }
GroupedKernelFn grouped_ring_f32_wide_ld(int combo) { return ring_wide_ld_kernel<float>(combo); }
}  // namespace jb
