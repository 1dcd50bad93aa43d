// Instances of the kernel with activations in registers (w4a16_regs_kernel.h): 4-bit codes in groups of 32 rows.
#include "w4a16_regs_kernel.h"

namespace vaq {
int regs_launch_w4_sub4(const RegsParams& p, int nw, int j, int mb, bool bf16, bool zp, hipStream_t s) {
  return zp ? regs_types<4, false, true>(p, nw, j, mb, bf16, s) : regs_types<4, false, false>(p, nw, j, mb, bf16, s);
}
}  // namespace vaq
