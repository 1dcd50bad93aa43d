// Instances of the 256 x 256 tile kernel (w4a16_tile256_kernel.h) for 4-bit codes in groups of 128 rows / channelwise.
#include "w4a16_tile256_kernel.h"

namespace vaq {

int prefill_launch_tile256(const PrefillParams& p, bool bf16, bool zp, hipStream_t s) {
  if (bf16) return zp ? launch_tile256<true, true, 1, false>(p, s) : launch_tile256<true, false, 1, false>(p, s);
  return zp ? launch_tile256<false, true, 1, false>(p, s) : launch_tile256<false, false, 1, false>(p, s);
}

}  // namespace vaq
