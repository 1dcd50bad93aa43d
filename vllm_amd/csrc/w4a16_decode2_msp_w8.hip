// Instances of the LDS-staged decode kernel with the rows split over workgroups for 8-bit codes, any group size.
#include "w4a16_decode2_kernel.h"

namespace vaq {

template <bool BF16, int SUBG>
static int msp_w8_dispatch(const Decode2Params& p, int gs, hipStream_t s) {
  switch (gs) {
    case 2: return launch_decode2<BF16, 2, 1, false, 16, SUBG, 1, 0, true>(p, s);
    case 4: return launch_decode2<BF16, 4, 1, false, 16, SUBG, 1, 0, true>(p, s);
    case 8: return launch_decode2<BF16, 8, 1, false, 16, SUBG, 1, 0, true>(p, s);
    case 14:
      if constexpr (SUBG == 1) return launch_decode2<BF16, 14, 1, false, 16, SUBG, 1, 0, true>(p, s);
      break;
    case 16: return launch_decode2<BF16, 16, 1, false, 16, SUBG, 1, 0, true>(p, s);
    default: break;
  }
  set_error("w4a16_gemm(decode, 8-bit): unsupported tiles per wavefront %d", gs);
  return VAQ_ERR_UNSUPPORTED;
}

int decode2_launch_msp_w8(const Decode2Params& p, int sub, int gs, bool bf16, hipStream_t s) {
  if (sub == 1) return bf16 ? msp_w8_dispatch<true, 1>(p, gs, s) : msp_w8_dispatch<false, 1>(p, gs, s);
  if (sub == 2) return bf16 ? msp_w8_dispatch<true, 2>(p, gs, s) : msp_w8_dispatch<false, 2>(p, gs, s);
  return bf16 ? msp_w8_dispatch<true, 4>(p, gs, s) : msp_w8_dispatch<false, 4>(p, gs, s);
}

}  // namespace vaq
