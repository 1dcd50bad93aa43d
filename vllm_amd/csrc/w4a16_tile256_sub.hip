// Instances of the 256 x 256 tile kernel (w4a16_tile256_kernel.h) for 4-bit codes in groups of 64 and 32 rows (2 / 4 per 128-row tile).
#include "w4a16_tile256_kernel.h"

namespace vaq {

template <int SUBG>
static int tile256_sub(const PrefillParams& p, bool bf16, bool zp, hipStream_t s) {
  if (bf16) return zp ? launch_tile256<true, true, SUBG, false>(p, s) : launch_tile256<true, false, SUBG, false>(p, s);
  return zp ? launch_tile256<false, true, SUBG, false>(p, s) : launch_tile256<false, false, SUBG, false>(p, s);
}

int prefill_launch_tile256_sub(const PrefillParams& p, int sub, bool bf16, bool zp, hipStream_t s) {
  return sub == 2 ? tile256_sub<2>(p, bf16, zp, s) : tile256_sub<4>(p, bf16, zp, s);
}

}  // namespace vaq
