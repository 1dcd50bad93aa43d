// Instances of the 256 x 256 tile kernel (w4a16_tile256_kernel.h) for 8-bit codes (groups of 128, 64 and 32 rows, channelwise).
#include "w4a16_tile256_kernel.h"

namespace vaq {

template <int SUBG>
static int tile256_w8(const PrefillParams& p, bool bf16, hipStream_t s) {
  return bf16 ? launch_tile256<true, false, SUBG, true>(p, s) : launch_tile256<false, false, SUBG, true>(p, s);
}

int prefill_launch_tile256_w8(const PrefillParams& p, int sub, bool bf16, hipStream_t s) {
  return sub == 1 ? tile256_w8<1>(p, bf16, s) : sub == 2 ? tile256_w8<2>(p, bf16, s) : tile256_w8<4>(p, bf16, s);
}

}  // namespace vaq
