// Instances of the strip kernel (w4a16_strip_kernel.h) for 8-bit codes (groups of 128, 64 and 32 rows, channelwise).
#include "w4a16_strip_kernel.h"

namespace vaq {

int prefill_launch_strip_w8(const PrefillParams& p, int sub, int tile, bool bf16, hipStream_t s) {
  switch (sub) {
    case 1: return bf16 ? strip_dispatch<true, false, 1, true>(p, tile, s) : strip_dispatch<false, false, 1, true>(p, tile, s);
    case 2: return bf16 ? strip_dispatch<true, false, 2, true>(p, tile, s) : strip_dispatch<false, false, 2, true>(p, tile, s);
    default: return bf16 ? strip_dispatch<true, false, 4, true>(p, tile, s) : strip_dispatch<false, false, 4, true>(p, tile, s);
  }
}

}  // namespace vaq
