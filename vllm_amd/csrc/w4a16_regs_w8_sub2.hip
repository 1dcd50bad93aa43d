// Instances of the kernel with activations in registers (w4a16_regs_kernel.h): 8-bit codes in groups of 64 rows.
#include "w4a16_regs_kernel.h"

namespace vaq {
int regs_launch_w8_sub2(const RegsParams& p, int nw, int j, int mb, bool bf16, hipStream_t s) {
  return regs_types<2, true, false>(p, nw, j, mb, bf16, s);
}
}  // namespace vaq
