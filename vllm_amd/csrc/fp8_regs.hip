// Host side of the FP8 GEMM for some dozen rows (fp8_regs_kernel.h): price of a plan, launch.
#include "fp8_regs_kernel.h"

#include <math.h>

namespace vaq {

// In us: `base`, `out` per MB of results; a workgroup `round`, `meet` for each 16 x 16 result and its steps, each the latency, the bytes into the compute unit or the
// products of all workgroups on it, whichever is longest, more where K is a multiple of 1024 (rows start on the same memory channels); beside that the weights
// from memory, `again` of them for every further block of rows.  Fitted to the cold times of 772 problems (profiles/plan_prices/fp8_some_rows.csv.gz; 1 .. 256 rows) with all their
// plans: 7 % rms, the cheapest plan takes 1.005 of the fastest one's time in the mean.  Rows that do not start with a cache line, K no multiple of 128: 1.00 of that up to
// K = 2048, 1.13 to 8192, 1.31 beyond (50 calls; 12080 x 1536 at M = 33 14.3 us, 12032 x 1536 10.5).
static double plan_us(int mb, int j, double M, double N, double K, int cus) {
  const double rb = ceil(M / (16 * mb)), per_cu = ceil(ceil(N / 16 / j) * rb / cus);
  const double slots = fmin(floor(160.0 * 1024 / fp8_regs_lds_bytes(mb, j)), 4.0), side = fmin(per_cu, slots), rounds = fmax(per_cu / slots, 1.0);
  const double steps = ceil(ceil(K / FP8_REGS_STEP) / FP8_REGS_WAVES), bytes = 0.0119 * 16 * side * (mb + j), work = 0.102 * side * mb * j;
  const double step = cbrt(0.122 + bytes * bytes * bytes + work * work * work) * ((int64_t)K % 1024 == 0 ? 1.077 : 1.0);
  const double core = rounds * (0.272 + steps * step + 0.0906 * mb * j), mem = 0.183e-6 * K * N * (1 + 0.338 * (rb - 1));
  const double us = 1.66 + cbrt(core * core * core + mem * mem * mem) + 0.258 * 2e-6 * M * N;
  return (int64_t)K % 128 != 0 ? us * (1 + 0.026 * K / 1024) : us;
}

Fp8RegsPlan fp8_regs_plan(int M, int N, int K) {
  Fp8RegsPlan best;
  const int cus = num_cus_current_device();
  for (int mb = 1; mb <= 4 && (mb == 1 || M > 16 * (mb - 1)); ++mb)
    for (int j = 1; j <= 4; ++j) {
      if (!fp8_regs_built(mb, j)) continue;
      const double us = plan_us(mb, j, M, N, K, cus);
      if (best.us < 0 || us < best.us) {
        best.mb = mb;
        best.j = j;
        best.us = us;
      }
    }
  return best;
}

template <bool BF16_OUT, int MB, int J, bool TAIL>
static bool launch(const Fp8MMParams& p_in, hipStream_t s) {
  Fp8MMParams p = p_in;
  const uint32_t NT = (uint32_t)p.N / 16, RB = ((uint32_t)p.M + MB * 16 - 1) / (MB * 16), ranges = (NT + J - 1) / J, per_xcd = (ranges * RB + 7) / 8;
  p.a_extent = (uint32_t)((int64_t)(p.M - 1) * p.lda + p.K);
  p.b_extent = (uint32_t)((int64_t)(p.N - 1) * p.ldb + p.K);
  constexpr size_t lds = fp8_regs_lds_bytes(MB, J);
  auto kern = fp8_mm_regs_kernel<BF16_OUT, MB, J, TAIL>;
  static size_t reserved[VAQ_MAX_DEVICES];
  if (reserve_dynamic_lds(reinterpret_cast<const void*>(kern), lds, reserved, "fp8_scaled_mm") != VAQ_OK) return false;
  const uint32_t steps = ((uint32_t)p.K + FP8_REGS_STEP - 1) / FP8_REGS_STEP, rest = (uint32_t)p.K % FP8_REGS_STEP;
  hipLaunchKernelGGL(kern, dim3(per_xcd * 8), dim3(FP8_REGS_WAVES * 64), lds, s,
                     (v8u{ptr_lo(p.a), ptr_hi(p.a), ptr_lo(p.b), ptr_hi(p.b), (uint32_t)p.lda, (uint32_t)p.ldb, p.a_extent, p.b_extent}),
                     (v4u{steps << 8 | rest, (uint32_t)p.M | RB << 16, ranges, per_xcd}), (v2u{NT, fp8_regs_magic(RB)}), p);
  return true;
}

template <bool BF16_OUT, int MB, int J>
static bool launch(const Fp8MMParams& p, hipStream_t s) {
  if constexpr (!fp8_regs_built(MB, J)) return false;
  else return p.K % FP8_REGS_STEP != 0 ? launch<BF16_OUT, MB, J, true>(p, s) : launch<BF16_OUT, MB, J, false>(p, s);
}

template <bool BF16_OUT, int MB>
static bool launch_mb(const Fp8MMParams& p, int j, hipStream_t s) {
  switch (j) {
    case 1: return launch<BF16_OUT, MB, 1>(p, s);
    case 2: return launch<BF16_OUT, MB, 2>(p, s);
    case 3: return launch<BF16_OUT, MB, 3>(p, s);
    case 4: return launch<BF16_OUT, MB, 4>(p, s);
    default: return false;
  }
}

template <bool BF16_OUT>
static bool launch_type(const Fp8MMParams& p, int mb, int j, hipStream_t s) {
  switch (mb) {
    case 1: return launch_mb<BF16_OUT, 1>(p, j, s);
    case 2: return launch_mb<BF16_OUT, 2>(p, j, s);
    case 3: return launch_mb<BF16_OUT, 3>(p, j, s);
    case 4: return launch_mb<BF16_OUT, 4>(p, j, s);
    default: return false;
  }
}

bool fp8_regs_launch(const Fp8MMParams& p, bool bf16, int mb, int j, hipStream_t s) {
  return bf16 ? launch_type<true>(p, mb, j, s) : launch_type<false>(p, mb, j, s);
}

}  // namespace vaq
