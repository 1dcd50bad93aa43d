// FP8 linear layer of a few rows in one launch: the weight-streaming GEMM (fp8_stream2_kernel.h) on activations that it
// quantises itself.  As two launches the quantisation of a few rows costs 2-3 us -- a launch and a chain of load, reduction
// and store -- while the memory system, which bounds the GEMM, stands idle.  Here every workgroup quantises all M rows,
// each wavefront its own K slab, after it has requested its first weights.  That repeats the arithmetic in every
// workgroup, so it pays while the rows are few.  Cold weights, two launches -> one, per token, M = 1 / 4 / 8: 4096 x 6144
// 9.1 / 9.3 / 9.5 -> 7.1 / 7.9 / 9.2 us, 4096 x 4096 7.7 / 8.0 / 8.3 -> 5.1 / 6.3 / 7.9 us, 4096 x 28672 24.1 / 23.6 / 23.9 ->
// 20.9 / 20.5 / 21.6 us, 14336 x 4096 at M = 1 / 4 15.6 / 16.5 -> 12.1 / 15.0 us, 2048 x 2048 5.5 / 5.6 / 5.9 -> 3.6 / 4.2 / 5.0 us.
// Not kept: the rows dealt out to all wavefronts of the workgroup and exchanged through LDS (two more barriers, 2 us).
#include "fp8_stream2_kernel.h"

#include <type_traits>

namespace vaq {

template <bool BF16, int KS, int MQ, bool STATIC>
static int launch_quant_mm(const Fp8MMParams& p_in, int wk, int gx, hipStream_t s) {
  constexpr int NSR = KS == 4 ? 2 : 4;
  Fp8MMParams p = p_in;
  p.nt_base = (p.N / 16) / gx;
  p.nt_rem = (p.N / 16) % gx;
  p.a_extent = (uint32_t)(((int64_t)(p.M - 1) * p.lda + p.K) * 2);
  p.b_extent = (uint32_t)((int64_t)(p.N - 1) * p.ldb + p.K);
  const size_t lds = (size_t)wk * NSR * 4096 + (wk > 1 ? (size_t)2 * wk * 1024 : 0) + (size_t)wk * MQ * 128;
  auto kern = fp8_mm_stream2_kernel<BF16, KS, 1, NSR, MQ, STATIC>;
  static size_t reserved[VAQ_MAX_DEVICES];
  if (const int rc = reserve_dynamic_lds(reinterpret_cast<const void*>(kern), lds, reserved, "fp8_quant_scaled_mm"); rc != VAQ_OK) return rc;
  launch_fp8_stream(kern, dim3(gx), wk, lds, s, p);
  return VAQ_OK;
}

template <bool BF16, int KS, bool STATIC>
static int dispatch_rows(const Fp8MMParams& p, int wk, int gx, hipStream_t s) {
  if (p.M == 1) return launch_quant_mm<BF16, KS, 1, STATIC>(p, wk, gx, s);
  if (p.M == 2) return launch_quant_mm<BF16, KS, 2, STATIC>(p, wk, gx, s);
  if constexpr (KS <= 8) {
    if (p.M > 4) return launch_quant_mm<BF16, KS, 8, STATIC>(p, wk, gx, s);
  }
  return launch_quant_mm<BF16, KS, 4, STATIC>(p, wk, gx, s);
}

// K steps (of 128) per wavefront, 0 where two launches are at least as fast.  From 10700 problems drawn over M = 1 .. 8,
// K = 1024 .. 16384, N = 1024 .. 28672 with cold weights, every choice timed (two launches against this one, geometric means:
// M = 1 1.28, M = 2 1.27, M = 3, 4 1.14 per token and 1.24 with a given scale, M = 5 .. 8 1.09 and 1.18 where taken; the
// choices below are on average 0.4 % from the best of each problem):
//  * 4 steps, that is more wavefronts for the quantisation: K <= 2048 (against 8 steps 4-10 % at M = 1, 14-30 % at M = 8), and
//    K <= 4096 with two rows and more (0-20 %), though not for up to four rows of a K <= 3072 on a layer of four rounds and
//    more of workgroups (8 steps 3-5 % ahead);
//  * 16 steps, a longer stream for each of fewer wavefronts: where 8 wavefronts of 8 steps do not cover K, and from K = 4097 on
//    for one row of more than a round (3-4 %) and two rows of more than three (1-3 %);
//  * per token, M > 4 up to K = 4096 only (K = 4100 .. 8000: 1-15 % slower than two launches); no M > 4 with 16 steps, whose
//    registers are full.
static int quant_mm_steps(int64_t M, int64_t N, int64_t K, bool per_token) {
  // (the kernel addresses the weights with 32-bit offsets: they end below 2 GiB whatever the row stride)
  if (M < 1 || M > 8 || K % 16 != 0 || N % 16 != 0 || N >= (1ll << 31) || K >= (1ll << 31) || N * K >= (1ll << 31)) return 0;
  const int64_t steps = (K + 127) / 128, NT = N / 16, cus = num_cus_current_device();
  if (steps <= 16) return 4;
  if (steps <= 32) return M == 1 || (M <= 4 && NT >= 4 * cus && steps <= 24) ? 8 : 4;
  if (steps <= 64 && M > 4) return per_token ? 0 : 8;
  if (steps < 64) return (M == 1 && NT > cus) || (M == 2 && NT > 3 * cus) ? 16 : 8;
  return steps <= 128 && M <= 4 ? 16 : 0;
}

// Workgroups: one per compute unit, except two of a short K (few wavefronts each) on layers of more than three rounds (K <= 2048
// 5-15 % ahead; per token and M > 4 up to K = 3072, 4 %), for K <= 1536 and up to four rows on more than one (0-5 %).
static int quant_mm_grid(int M, int NT, int steps, int ks, bool per_token) {
  const int cus = num_cus_current_device();
  const bool two = ks == 4 && ((NT > 3 * cus && (steps <= 16 || (steps <= 24 && per_token && M > 4))) || (NT > cus && steps <= 12 && M <= 4));
  const int slots = two ? 2 * cus : cus, rounds = (NT + slots - 1) / slots;
  return (NT + rounds - 1) / rounds;
}

}  // namespace vaq

extern "C" int vaq_fp8_quant_scaled_mm_takes(int64_t size_m, int64_t size_n, int64_t size_k, int per_token) {
  return vaq::quant_mm_steps(size_m, size_n, size_k, per_token != 0) != 0;
}

extern "C" int vaq_fp8_quant_scaled_mm(const void* x, int64_t ldx, const float* x_scale, const uint8_t* b, int64_t ldb, const float* sb,
                                       int64_t sb_count, const void* bias, void* out, int64_t ldc, int dtype, int64_t size_m,
                                       int64_t size_n, int64_t size_k, void* stream) {
  using namespace vaq;
  const char* const who = "fp8_quant_scaled_mm";
  VAQ_CHECK_ARG(size_m >= 0 && size_n > 0 && size_k > 0, "%s: bad shape M=%lld N=%lld K=%lld", who, (long long)size_m,
                (long long)size_n, (long long)size_k);
  VAQ_CHECK_ARG(dtype == VAQ_F16 || dtype == VAQ_BF16, "%s: dtype tag %d", who, dtype);
  VAQ_CHECK_ARG(ldx >= size_k && ldx % 8 == 0, "%s: x row stride %lld must be >= K and a multiple of 8", who, (long long)ldx);
  VAQ_CHECK_ARG(ldb >= size_k && ldb % 16 == 0, "%s: b column stride %lld must be >= K and a multiple of 16", who, (long long)ldb);
  VAQ_CHECK_ARG(ldc >= size_n && ldc % 8 == 0, "%s: out row stride %lld must be >= N and a multiple of 8", who, (long long)ldc);
  VAQ_CHECK_ARG(sb_count == 1 || sb_count == size_n, "%s: b_scales count %lld must be 1 or N", who, (long long)sb_count);
  if (size_m == 0) return VAQ_OK;
  const int ks = quant_mm_steps(size_m, size_n, size_k, x_scale == nullptr);
  VAQ_CHECK_SUPPORTED(ks != 0 && (size_m - 1) * ldx + size_k < (1ll << 30) && (size_n - 1) * ldb + size_k < (1ll << 31),
                      "%s: M=%lld N=%lld K=%lld is quantised and multiplied by two kernels", who, (long long)size_m, (long long)size_n,
                      (long long)size_k);
  VAQ_CHECK_ARG(x && b && sb && out, "%s: null pointer", who);
  VAQ_CHECK_ARG(((uintptr_t)x % 16) == 0 && ((uintptr_t)b % 16) == 0 && ((uintptr_t)out % 8) == 0,
                "%s: x and b must be 16-byte aligned, out 8-byte aligned", who);
  VAQ_CHECK_ARG(((uintptr_t)sb % 16) == 0 && (!bias || ((uintptr_t)bias % 8) == 0),
                "%s: b_scales must be 16-byte aligned, bias 8-byte aligned", who);
  Fp8MMParams p;
  p.a = (const uint8_t*)x; p.lda = ldx; p.b = b; p.ldb = ldb;
  p.sa = x_scale; p.sa_per_row = 0;
  p.sb = sb; p.sb_per_col = (sb_count > 1 || size_n == 1) ? 1 : 0;
  p.bias = (const uint16_t*)bias;
  p.out = (uint16_t*)out; p.ldc = ldc;
  p.M = (int)size_m; p.N = (int)size_n; p.K = (int)size_k;
  const int steps = (p.K + 127) / 128, NT = p.N / 16;
  const int wk = (steps + ks - 1) / ks;
  const int gx = quant_mm_grid(p.M, NT, steps, ks, x_scale == nullptr);
  hipStream_t s = (hipStream_t)stream;
  auto run = [&](auto bf16_c, auto static_c) {
    constexpr bool B = decltype(bf16_c)::value, S = decltype(static_c)::value;
    return ks == 4 ? dispatch_rows<B, 4, S>(p, wk, gx, s) : (ks == 8 ? dispatch_rows<B, 8, S>(p, wk, gx, s) : dispatch_rows<B, 16, S>(p, wk, gx, s));
  };
  using TT = std::true_type;
  using FF = std::false_type;
  const int rc = dtype == VAQ_BF16 ? (x_scale ? run(TT{}, TT{}) : run(TT{}, FF{})) : (x_scale ? run(FF{}, TT{}) : run(FF{}, FF{}));
  if (rc != VAQ_OK) return rc;
  VAQ_CHECK_LAUNCH("fp8_quant_scaled_mm");
  return VAQ_OK;
}
