// Instances of the strip kernel (w4a16_strip_kernel.h) for 4-bit codes in groups of 64 and 32 rows (2 / 4 per 128-row tile).
#include "w4a16_strip_kernel.h"

namespace vaq {

template <int SUBG>
static int strip_sub(const PrefillParams& p, int tile, bool bf16, bool zp, hipStream_t s) {
  if (bf16) return zp ? strip_dispatch<true, true, SUBG, false>(p, tile, s) : strip_dispatch<true, false, SUBG, false>(p, tile, s);
  return zp ? strip_dispatch<false, true, SUBG, false>(p, tile, s) : strip_dispatch<false, false, SUBG, false>(p, tile, s);
}

int prefill_launch_strip_sub(const PrefillParams& p, int sub, int tile, bool bf16, bool zp, hipStream_t s) {
  return sub == 2 ? strip_sub<2>(p, tile, bf16, zp, s) : strip_sub<4>(p, tile, bf16, zp, s);
}

}  // namespace vaq
