// Instances of the LDS-staged decode kernel with the rows split over workgroups for 4-bit codes in groups of 64 / 32 rows.
#include "w4a16_decode2_kernel.h"

namespace vaq {

template <bool BF16, bool HAS_ZP, int SUBG>
static int msp_sub_dispatch(const Decode2Params& p, int gs, hipStream_t s) {
  switch (gs) {
    case 1: return launch_decode2<BF16, 1, 1, HAS_ZP, 16, SUBG, 0, 0, true>(p, s);
    case 2: return launch_decode2<BF16, 2, 1, HAS_ZP, 16, SUBG, 0, 0, true>(p, s);
    case 4: return launch_decode2<BF16, 4, 1, HAS_ZP, 16, SUBG, 0, 0, true>(p, s);
    case 8: return launch_decode2<BF16, 8, 1, HAS_ZP, 16, SUBG, 0, 0, true>(p, s);
    case 16: return launch_decode2<BF16, 16, 1, HAS_ZP, 16, SUBG, 0, 0, true>(p, s);
    default: break;
  }
  set_error("w4a16_gemm(decode): unsupported groups per wavefront %d", gs);
  return VAQ_ERR_UNSUPPORTED;
}

template <int SUBG>
static int msp_sub_types(const Decode2Params& p, int gs, bool bf16, bool zp, hipStream_t s) {
  if (bf16) return zp ? msp_sub_dispatch<true, true, SUBG>(p, gs, s) : msp_sub_dispatch<true, false, SUBG>(p, gs, s);
  return zp ? msp_sub_dispatch<false, true, SUBG>(p, gs, s) : msp_sub_dispatch<false, false, SUBG>(p, gs, s);
}

int decode2_launch_msp_sub(const Decode2Params& p, int sub, int gs, bool bf16, bool zp, hipStream_t s) {
  return sub == 2 ? msp_sub_types<2>(p, gs, bf16, zp, s) : msp_sub_types<4>(p, gs, bf16, zp, s);
}

}  // namespace vaq
