// Instances of the strip kernel (w4a16_strip_kernel.h) for 4-bit codes in groups of 128 rows / channelwise.
#include "w4a16_strip_kernel.h"

namespace vaq {

int prefill_launch_strip(const PrefillParams& p, int tile, bool bf16, bool zp, hipStream_t s) {
  if (bf16) return zp ? strip_dispatch<true, true, 1, false>(p, tile, s) : strip_dispatch<true, false, 1, false>(p, tile, s);
  return zp ? strip_dispatch<false, true, 1, false>(p, tile, s) : strip_dispatch<false, false, 1, false>(p, tile, s);
}

}  // namespace vaq
