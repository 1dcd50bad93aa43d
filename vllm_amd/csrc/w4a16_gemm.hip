// C-ABI entry of the W4A16 GEMM: argument validation and the decode / prefill dispatch.
#include "tile_plan.h"
#include "w4a16_kernels.h"

#include <mutex>

namespace vaq {

constexpr int64_t DECODE_MAX_M = 64;          // up to four m-blocks of 16 rows on the LDS-staged kernel
constexpr int64_t DECODE_MAX_M_2BLK = 32;     // the register-resident kernel, groups below 128 rows and 8-bit codes: two

// Measured on MI355X (cold weights): staging the activations once per workgroup in LDS (one independent task per
// wavefront, no barrier in the K loop) wins on every Llama-3-8B projection and on 8192 x 28672 (30 us against 43.5 us
// for 3 <= M <= 16).  The register-resident kernel, whose wavefronts walk over n-tiles with their slice of the
// activations held in registers, stays ahead only on a vocabulary-sized layer (4096 x 128256, 3 <= M <= 16: 55 us
// against 62 us).
static int decode_impl_for(int64_t size_m, int64_t size_n, int64_t lda, int sub, bool w8) {
  // the LDS-staged kernel addresses A through a 32-bit buffer offset
  if (size_m * lda * 2 >= (1ll << 31)) return 1;
  if (sub > 1 || w8) return 0;    // groups below 128 rows and 8-bit codes are built for the LDS-staged kernel only
  if (tuning().decode_impl > 0) return tuning().decode_impl - 1;   // tests / benchmarks: 1 LDS-staged, 2 register-resident
  return (size_n >= 65536 && size_m > 2 && size_m <= 16) ? 1 : 0;
}

static int check_shape(int64_t size_m, int64_t size_n, int64_t size_k) {
  VAQ_CHECK_ARG(size_m >= 0, "w4a16_gemm: size_m = %lld is negative", (long long)size_m);
  VAQ_CHECK_ARG(size_n > 0 && size_n % 64 == 0, "w4a16_gemm: size_n = %lld, is not divisible by min_thread_n = 64",
                (long long)size_n);
  VAQ_CHECK_ARG(size_k > 0 && size_k % 128 == 0, "w4a16_gemm: size_k = %lld, is not divisible by min_thread_k = 128",
                (long long)size_k);
  VAQ_CHECK_ARG(size_m < (1ll << 31) && size_n < (1ll << 31) && size_k < (1ll << 31) &&
                    size_k * size_n / 2 < (1ll << 32),
                "w4a16_gemm: problem too large");   // (8-bit weights: K*N bytes, still below 2^33; offsets are checked per kernel)
  return VAQ_OK;
}

// Weight type tag and group size -> 4-bit (0), 8-bit (1) or FP8 (2) weights, groups per 128 rows, channelwise scales or not.
static int check_format(int64_t size_k, int group_size, int wtype, int* wt, int* sub, bool* channelwise) {
  VAQ_CHECK_ARG(wtype == VAQ_WTYPE_U4B8 || wtype == VAQ_WTYPE_U4 || wtype == VAQ_WTYPE_U8B128 || wtype == VAQ_WTYPE_FE4M3,
                "w4a16_gemm: unknown weight type tag %d", wtype);
  *wt = wtype == VAQ_WTYPE_U8B128 ? 1 : (wtype == VAQ_WTYPE_FE4M3 ? 2 : 0);
  *channelwise = group_size == -1 || (group_size == size_k && size_k != 128);
  VAQ_CHECK_SUPPORTED(*channelwise || group_size == 128 || group_size == 64 || group_size == 32,
                      "w4a16_gemm: group_size = %d is not built (only -1, 32, 64, 128)", group_size);
  *sub = *channelwise ? 1 : 128 / group_size;
  return VAQ_OK;
}

// What takes a problem of up to 256 rows where the kernel with activations in registers does not, and its predicted time; with `act_order` beyond 32 rows, the columns
// permuted: workgroups of 16 rows take few of those (w4a16_decode2_choose).
static int other_kind(int M, int N, int K, int sub, int wt, bool act_order, double* us) {
  const bool w8 = wt != 0, plain = sub == 1 && !w8;
  int kind = D2_WORKGROUP;
  // 3 .. 16 rows of a vocabulary-sized layer: the register-resident kernel.  A launch, for every 1000 columns its walk, the weights, and those times the
  // rows, and a hand-over for each started 4096 rows of K beyond the first; 10 % rms over 7.4e4 timings of K 256 .. 20480, N 65536 .. 152064.
  if (decode_impl_for(M, N, K, sub, w8) == 1) {
    *us = 3.08 + N * 1e-3 * (0.152 + K / 1024.0 * (0.0654 + 0.0084 * M / 16) + 0.556 * ((K + 4095) / 4096 - 1));
    return kind;
  }
  if (M > 16) {
    const int most = !plain ? DECODE_MAX_M_2BLK : N > 8192 ? 48 : DECODE_MAX_M;
    kind = w4a16_decode2_choose(M, N, K, sub, wt, act_order && M > DECODE_MAX_M_2BLK, false, M <= most, true, w4a16_staged_us(M, N, K, plain));
  }
  *us = kind == D2_TILE ? w4a16_tile_us(M, N, K, tile_format(sub, wt)) : w4a16_decode2_us(M, N, K, sub, w8, kind == D2_ROWS);
  return kind;
}

// Whether the kernel with activations in registers takes a problem: where its price is below this share of the price of what takes it otherwise.  The
// prices are older than the arguments in registers and off by as much as the kernels have gained since (this one's 3-5 % low, that of the decode kernel 0-8 % low
// with 4-bit codes in groups of 128 rows and 3-15 % low with the rest), so the shares are set by the choices, for one, 2 .. 4, 5 .. 16, 17 .. 32, 33 .. 64
// and more rows: over 3575 problems of random layers with both timed now the choice takes 1.010 of the faster one's time in the mean.  The shares before (0.85 up
// to 4 rows and 0.91 up to 32 for 4-bit codes in groups of 128 rows, 0.95 up to 32 for groups of 64 / 32) took 1.016.  (One row of those: 0.85 still, the decode
// kernel's instance for it is up to 27 % cheaper than priced; 4096 x 28672 11.9 us there, priced 15.1, and 12.8 here.)  Drawn layers: 9216 x
// 4416 at M = 4 9.2 -> 8.0 us, 11520 x 5248 at M = 18 14.0 -> 12.9; 1792 x 11008 at M = 3 4.5 -> 4.9.  From 33 rows on shares nearer to one lose as much as they gain: strips cost less, and zero points in small groups more, than priced (4-bit
// codes in groups of 32 with zero points at M = 34 13.7 -> 15.7).
static double regs_lead(int M, int N, int K, int sub, int wt, int j, int nw) {
  constexpr double SHARE[4][6] = {{0.85, 0.95, 0.96, 0.97, 0.95, 0.92}, {1.05, 1.05, 1.0, 1.0, 0.88, 0.88}, {1.05, 1.05, 1.0, 0.95, 0.88, 0.88},
                                  {1.17, 1.17, 1.01, 1.01, 0.95, 0.95}};
  // vocabulary-sized layers at 3 .. 16 rows, where another kernel is the alternative (it takes them all: 0.37 .. 0.96 of the time, 1 of 2000 more than 3 % slower;
  // 4096 x 128256 at M = 4 / 16 54.9 / 59.0 -> 51.9 / 53.4 us, 1024 x 128256 33.4 / 34.0 -> 18.1 / 19.5, 5120 x 65536 80.0 / 81.0 -> 33.2 / 34.7)
  if (wt == 0 && decode_impl_for(M, N, K, sub, false) == 1) return 0.95;
  double lead = SHARE[wt != 0 ? 3 : sub == 1 ? 0 : sub == 2 ? 1 : 2][M <= 1 ? 0 : M <= 4 ? 1 : M <= 16 ? 2 : M <= 32 ? 3 : M <= 64 ? 4 : 5];
  if (wt != 0 || sub > 1 || M > 32) return lead;
  // One n-tile to a wavefront, N from 2048 on, at 2 .. 4 rows: where eight slices of four or of eight k-tiles fill K to nine tenths the decode kernel's plan leaves nobody idle and is up to
  // 13 % cheaper than priced.  333 problems of K 3200 .. 8192, both timed: at 0.95 the choice takes 1.019 of the faster one's time and 79 calls here are more than 3 % slower
  // (7040 x 2560 at M = 2 5.7 us, 5.0 there); so 1.004 and 12, the 83 that go back take 0.942 of their time, one 1.05.
  const int tiles = K / 128;
  if (M > 1 && M <= 4 && j == 1 && N >= 2048 && ((tiles > 28 && tiles <= 32) || (tiles > 49 && tiles <= 64)) && lead > 0.84) lead = 0.84;
  // Where this kernel loses most of what it loses, by as much as the two prices together are off by: K of whole 1024 rows; one n-tile to a wavefront and K
  // beyond 8192 at up to 4 rows; two and more n-tiles on a short K.  Off are: this kernel's price, which counts 16 rows to a block, by the rows that a block has;
  // for workgroups of four; for one n-tile, which leaves 2 KB of weights in flight, by how much of the device waits for them and how long; for three and more
  // on a short K; the other's by what it fetches for one to four rows.  Fitted to 60520 + 860 timings of either, 6.6 % rms.  Over 33847 random ones
  // 2.0 -> 1.2 % of the calls lose more than 3 % (ordinary K and N, 75288: 2.5 -> 0.8); 1.4 % (3.2) go back to the decode kernel, 2.6 % ahead on them in the
  // mean: 4096 x 4096 at M = 16 5.5 -> 5.3 us, 2048 x 10240 6.1 -> 5.6, 11008 x 4096 at M = 1 8.4 -> 7.7, 13824 x 3584 at M = 2 9.6 -> 8.8.  Asked of
  // every K and plan it would send back as many that gain (K = 1152 .. 1536: +10 %).
  if (!(K % 1024 == 0 || (M <= 4 && j == 1 && K > 8192) || (K <= 2048 && ((j == 2 && K >= 1024) || (j >= 3 && K > 1536))))) return lead;
  const double lk = log2(K / 4096.0), full = j == 1 ? fmin(1.0, N / 16.0 / num_cus_current_device()) : 0;
  const double off = 0.031 + 0.109 * ((M - 1) % 16 + 1) / 16 + (M <= 4 ? 0.044 : 0) - (nw == 4 ? 0.061 : 0) - 0.019 * lk +
                     full * (0.038 + 0.075 * fmax(0.0, lk)) + (j >= 3 && K <= 2048 && N >= 4096 ? 0.046 : 0);
  const double by_price = exp(-0.01 - off);
  return lead < by_price ? lead : by_price;
}
bool w4a16_takes_regs(int M, int N, int K, int sub, int wt, double* other, bool act_order) {
  const TuningScope automatic(nullptr);
  int j = 0, nw = 0;
  const double us = w4a16_regs_us(M, N, K, sub, wt, &j, &nw);
  if (us < 0) return false;
  other_kind(M, N, K, sub, wt, act_order, other);
  return us < *other * regs_lead(M, N, K, sub, wt, j, nw);
}

// Whether a switch names a kernel or a plan of one.
static bool plan_named(const VaqTuning& tn) {
  return tn.decode_impl > 0 || tn.decode2_gs > 0 || tn.decode2_wks > 0 || tn.decode2_wn > 0 || tn.prefill_tile > 0 || tn.prefill_split > 0 ||
         tn.exp[0] > 0 || tn.exp[1] > 0 || tn.exp[2] > 0 || tn.exp[3] > 0 || tn.exp[5] > 0 || tn.exp[6] > 0;
}

// The same for a call, from a table per thread.  A switch that names another kernel or a plan of one keeps it out; exp[8] asks for it.
static bool regs_chosen(int M, int N, int K, int sub, int wt, bool act_order) {
  const VaqTuning& tn = tuning();
  if (M < 1 || M > REGS_MAX_M || N >= (1 << 24) || K >= (1 << 24) || tn.exp[8] == 1) return false;
  if (tn.exp[8] > 1) return w4a16_regs_us(M, N, K, sub, wt) >= 0;
  if (plan_named(tn)) return false;
  static thread_local PlanTable<int> table;
  double other;
  return table.get(M, N, K, (num_cus_current_device() * 8 + sub) * 8 + wt * 2 + act_order, [&] { return w4a16_takes_regs(M, N, K, sub, wt, &other, act_order) ? 1 : 0; }) != 0;
}

// Whether act_order's columns are permuted by a launch of their own ahead of the kernels with activations in registers and the decode kernels too,
// which then run as without act_order (the gather inside the decode kernel is two dependent loads per element, in every workgroup, and the kernel with
// activations in registers has none).  Beyond 32 rows always: 4096 x 4096 at M = 48 / 64 20.4 / 25.3 -> 9.7 / 10.2 us, 14336 x 4096 50 / 64 -> 21.1 / 21.8.
// Up to there where the gather is priced above 2 us (the launch takes 2.4 from one to the other) and the call above 8.6, which is what the host needs
// for a call of two launches (5.5 for one).  Over 1077 calls of drawn act_order layers of 1 .. 32 rows the 773 it takes run in 0.57 of their time in
// the mean, none slower; of the others 94 would gain more than a tenth replayed from a graph, 28 called.  4096 x 4096 at M = 8 / 16 / 32 12.5 / 20.7 / 23.2 -> 7.1 /
// 7.7 / 8.2 us, 14336 x 4096 at M = 1 / 16 12.1 / 39.3 -> 10.7 / 14.8, 9088 x 2560 in 8-bit codes at M = 16 31.3 -> 12.4; left as they are 4096 x 28672 at
// M = 1 13.6 (15.4), 2048 x 2048 at M = 4 5.7 (6.1) and 4096 x 4096 at M = 4 8.6 (6.6, and 8.5 for the host).  3 .. 16 rows of a vocabulary-sized layer, always: 4096 x 128256 at M = 4 61.1 -> 46.4 us.
static bool permutes_first(int M, int N, int K, int sub, bool w8) {
  const VaqTuning& tn = tuning();
  if (M < 1 || N >= (1 << 24) || K >= (1 << 24) || tn.exp[9] == 1 || plan_named(tn)) return false;
  if (M > DECODE_MAX_M_2BLK || decode_impl_for(M, N, K, sub, w8) == 1) return true;
  static thread_local PlanTable<int> table;
  return table.get(M, N, K, num_cus_current_device() * 8 + sub + (w8 ? 1 << 16 : 0), [&] {
    double gather = 0;
    const double us = w4a16_decode2_gather_us(M, N, K, sub, w8, &gather);
    return gather > 2.0 && us > 8.6 ? 1 : 0;
  }) != 0;
}

// Whether `bytes` of partial tiles and `ints` counters are enough for a call of up to 32 rows with act_order whose columns are permuted.
static bool small_call_fits(int M, int N, int K, int sub, int wt, int64_t bytes, int64_t ints) {
  size_t t = 0, n = 0;
  auto fits = [&] { return bytes >= (int64_t)t && ints >= (int64_t)n; };
  if (regs_chosen(M, N, K, sub, wt, true)) {
    w4a16_regs_workspace(M, N, K, sub, wt != 0, &t, &n);
    if (fits()) return true;
  }
  if (decode_impl_for(M, N, K, sub, wt != 0) == 1) w4a16_decode_workspace(M, N, K, &t, &n);
  else w4a16_decode2_workspace(M, N, K, sub, wt != 0, &t, &n);
  return fits();
}

// Scratch of a problem, enough for whichever kernel runs (that also depends on the row stride of A): for one weight format, or with
// wt < 0 for any of them.
static int scratch_of(int64_t size_m, int64_t size_n, int64_t size_k, bool has_perm, int wt, int sub, size_t* c_tmp_bytes,
                      size_t* a_tmp_bytes, size_t* counter_ints) {
  VAQ_CHECK_ARG(c_tmp_bytes && a_tmp_bytes && counter_ints, "w4a16_gemm_workspace: null output pointer");
  int rc = check_shape(size_m, size_n, size_k);
  if (rc != VAQ_OK) return rc;
  *c_tmp_bytes = 0;
  *a_tmp_bytes = 0;
  *counter_ints = 0;
  const int M = (int)size_m, N = (int)size_n, K = (int)size_k;
  auto take = [&](size_t t, size_t n) {
    if (t > *c_tmp_bytes) *c_tmp_bytes = t;
    if (n > *counter_ints) *counter_ints = n;
  };
  size_t t = 0, n = 0;
  for (int s : {1, 2, 4})
    for (bool w8 : {false, true}) {
      const bool plain = s == 1 && !w8;
      if (size_m > (plain ? DECODE_MAX_M : DECODE_MAX_M_2BLK) || size_m == 0 || (wt >= 0 && (s != sub || w8 != (wt != 0)))) continue;
      rc = w4a16_decode2_workspace(M, N, K, s, w8, &t, &n);
      if (rc != VAQ_OK) return rc;
      take(t, n);
      if (!plain || size_m > DECODE_MAX_M_2BLK) continue;
      rc = w4a16_decode_workspace(M, N, K, &t, &n);
      if (rc != VAQ_OK) return rc;
      take(t, n);
    }
  // from 17 rows on the tile kernel where it is ahead
  if (size_m > 16)
    for (TileFormat format : {TILES_PLAIN, TILES_SUB, TILES_8BIT, TILES_8BIT_64, TILES_8BIT_32, TILES_FP8}) {
      if (wt >= 0 && format != tile_format(sub, wt)) continue;
      rc = w4a16_prefill_workspace(M, N, K, format, &t, &n);
      if (rc != VAQ_OK) return rc;
      take(t, n);
    }
  size_t columns = 0;      // act_order: room for the permuted columns, behind the partial tiles up to 32 rows
  for (int s : {1, 2, 4})
    for (int w : {0, 1}) {
      if (size_m == 0 || (wt >= 0 && (s != sub || w != wt)) || (has_perm && !permutes_first(M, N, K, s, w == 1))) continue;
      if (has_perm && size_m <= DECODE_MAX_M_2BLK) columns = (size_t)size_m * (size_t)size_k * 2;
      if (size_m > REGS_MAX_M || !regs_chosen(M, N, K, s, w, has_perm)) continue;
      w4a16_regs_workspace(M, N, K, s, w == 1, &t, &n);
      take(t, n);
    }
  if (columns) *c_tmp_bytes = ((*c_tmp_bytes + 15) & ~(size_t)15) + columns;
  if (has_perm && size_m > DECODE_MAX_M_2BLK) *a_tmp_bytes = (size_t)size_m * (size_t)size_k * 2;
  return VAQ_OK;
}

// A checked call on the kernel that takes it.  `act_order` with `perm` null: the columns of A have been permuted.
static int dispatch(const void* a, int64_t lda, const int32_t* b, const void* scales, const int32_t* zeros, const int32_t* perm, bool act_order,
                    const void* bias, void* c, float* c_tmp, int64_t c_tmp_bytes, void* a_tmp, int32_t* counters, int64_t counter_ints,
                    int64_t size_m, int64_t size_n, int64_t size_k, int sub, bool channelwise, int wt, int dtype, int force_path, hipStream_t s) {
  const bool w8 = wt != 0;
  // The kernel with operands in registers first: a call that it takes looks up none of the other plans.  (One that brings too little scratch for its parts of K
  // goes on to the others; so does one whose rows end beyond 2 GiB.)
  if (force_path == 0 && perm == nullptr && size_m <= REGS_MAX_M && size_m * lda * 2 < (1ll << 31) &&
      regs_chosen((int)size_m, (int)size_n, (int)size_k, sub, wt, act_order)) {
    size_t t = 0, n = 0;
    w4a16_regs_workspace((int)size_m, (int)size_n, (int)size_k, sub, w8, &t, &n);
    if ((t == 0 && n == 0) || (c_tmp != nullptr && counters != nullptr && (uintptr_t)c_tmp % 16 == 0 && c_tmp_bytes >= (int64_t)t && counter_ints >= (int64_t)n))
      return w4a16_regs_launch(a, lda, b, scales, zeros, bias, c, c_tmp, counters, (int)size_m, (int)size_n, (int)size_k, sub, channelwise,
                               w8, dtype, s);
  }

  // three and four m-blocks exist on the LDS-staged kernel for 4-bit codes in groups of 128 rows / channelwise
  const bool two_blocks_only = sub > 1 || w8 || decode_impl_for(size_m, size_n, lda, sub, w8) != 0;
  // (measured: four m-blocks beat the tile kernel by 1.5-2x on the narrow layers and lose 3 % on a 28672-wide one)
  const int64_t dec_max = two_blocks_only ? DECODE_MAX_M_2BLK : (size_n > 8192 ? 48 : DECODE_MAX_M);
  bool decode = size_m <= dec_max, rows = false;
  VAQ_CHECK_ARG(force_path != 1 || decode, "w4a16_gemm: decode path forced with size_m = %lld > %lld", (long long)size_m,
                (long long)dec_max);
  if (force_path == 2) {
    decode = false;
  } else if (size_m > 16 && size_m <= 256 && size_n < (1 << 24) && size_k < (1 << 24) &&
             decode_impl_for(size_m, size_n, lda, sub, w8) == 0) {
    // 17 .. 256 rows: the decode kernel's workgroups of all rows or of 16 rows each, or the tile kernel (where it is given the
    // scratch that its plan asks for; up to 32 rows that need not be so, and act_order stays with the decode kernel)
    bool tile_ok = force_path == 0;
    if (tile_ok && size_m <= DECODE_MAX_M_2BLK) {
      size_t t = 0, n = 0;
      w4a16_prefill_workspace((int)size_m, (int)size_n, (int)size_k, tile_format(sub, wt), &t, &n);
      tile_ok = !act_order && c_tmp_bytes >= (int64_t)t && counter_ints >= (int64_t)n;
    }
    const int kind = w4a16_decode2_choose((int)size_m, (int)size_n, (int)size_k, sub, wt, act_order, perm != nullptr, decode, tile_ok || !decode,
                                          w4a16_staged_us((int)size_m, (int)size_n, (int)size_k, !w8 && sub == 1));
    decode = kind != D2_TILE;
    rows = kind == D2_ROWS;
  }
  if (decode && decode_impl_for(size_m, size_n, lda, sub, w8) == 0)
    return w4a16_decode2_launch(a, lda, b, scales, zeros, perm, bias, c, c_tmp, c_tmp_bytes, counters, counter_ints, (int)size_m,
                                (int)size_n, (int)size_k, sub, channelwise, wt, dtype, rows, s);
  if (decode) {
    VAQ_CHECK_SUPPORTED(sub == 1 && !w8, "w4a16_gemm: group_size = %d / 8-bit weights with an A of 2 GiB or more are not built",
                        channelwise ? -1 : 128 / sub);
    return w4a16_decode_launch(a, lda, b, scales, zeros, perm, bias, c, c_tmp, c_tmp_bytes, counters, counter_ints, (int)size_m,
                               (int)size_n, (int)size_k, channelwise, dtype, s);
  }

  const void* a_eff = a;
  int64_t lda_eff = lda;
  if (perm) {
    VAQ_CHECK_ARG(a_tmp != nullptr, "w4a16_gemm: act_order on the prefill path needs a_tmp [size_m, size_k]");
    VAQ_CHECK_ARG(((uintptr_t)a_tmp % 16) == 0, "w4a16_gemm: a_tmp must be 16-byte aligned");
    const int rc = vaq_permute_cols(a, lda, perm, a_tmp, size_m, size_k, s);
    if (rc != VAQ_OK) return rc;
    a_eff = a_tmp;
    lda_eff = size_k;
  }
  return w4a16_prefill_launch(a_eff, lda_eff, b, scales, zeros, bias, c, c_tmp, c_tmp_bytes, counters, counter_ints, (int)size_m,
                              (int)size_n, (int)size_k, sub, channelwise, wt, dtype, s);
}
}  // namespace vaq

extern "C" int vaq_w4a16_gemm_workspace_of_format(int64_t size_m, int64_t size_n, int64_t size_k, int group_size, int wtype,
                                                  int has_perm, int device, size_t* c_tmp_bytes, size_t* a_tmp_bytes,
                                                  size_t* counter_ints) {
  using namespace vaq;
  (void)device;
  int wt = 0, sub = 1;
  bool channelwise = false;
  int rc = check_shape(size_m, size_n, size_k);
  if (rc == VAQ_OK) rc = check_format(size_k, group_size, wtype, &wt, &sub, &channelwise);
  if (rc != VAQ_OK) return rc;
  return scratch_of(size_m, size_n, size_k, has_perm != 0, wt, sub, c_tmp_bytes, a_tmp_bytes, counter_ints);
}

extern "C" int vaq_w4a16_gemm_workspace(int64_t size_m, int64_t size_n, int64_t size_k, int has_perm, int device,
                                        size_t* c_tmp_bytes, size_t* a_tmp_bytes, size_t* counter_ints) {
  return vaq_w4a16_gemm_workspace_tuned(size_m, size_n, size_k, has_perm, device, c_tmp_bytes, a_tmp_bytes, counter_ints,
                                        nullptr);
}

extern "C" int vaq_w4a16_gemm_workspace_tuned(int64_t size_m, int64_t size_n, int64_t size_k, int has_perm, int device,
                                              size_t* c_tmp_bytes, size_t* a_tmp_bytes, size_t* counter_ints,
                                              const VaqTuning* tuning_or_null) {
  using namespace vaq;
  (void)device;
  const TuningScope scope(tuning_or_null);
  return scratch_of(size_m, size_n, size_k, has_perm != 0, -1, 0, c_tmp_bytes, a_tmp_bytes, counter_ints);
}

extern "C" int vaq_w4a16_gemm(const void* a, int64_t lda, const int32_t* b, const void* scales, const int32_t* zeros,
                              const int32_t* perm, const void* bias, void* c, float* c_tmp, int64_t c_tmp_bytes,
                              void* a_tmp, int32_t* counters, int64_t counter_ints, int64_t size_m, int64_t size_n,
                              int64_t size_k, int group_size, int dtype, int wtype, int force_path, void* stream) {
  return vaq_w4a16_gemm_tuned(a, lda, b, scales, zeros, perm, bias, c, c_tmp, c_tmp_bytes, a_tmp, counters, counter_ints,
                              size_m, size_n, size_k, group_size, dtype, wtype, force_path, stream, nullptr);
}

extern "C" int vaq_w4a16_gemm_tuned(const void* a, int64_t lda, const int32_t* b, const void* scales,
                                    const int32_t* zeros, const int32_t* perm, const void* bias, void* c, float* c_tmp,
                                    int64_t c_tmp_bytes, void* a_tmp, int32_t* counters, int64_t counter_ints,
                                    int64_t size_m, int64_t size_n, int64_t size_k, int group_size, int dtype, int wtype,
                                    int force_path, void* stream, const VaqTuning* tuning_or_null) {
  using namespace vaq;
  const TuningScope scope(tuning_or_null);
  VAQ_CHECK_ARG(c_tmp_bytes >= 0 && counter_ints >= 0, "w4a16_gemm: negative scratch size");
  int rc = check_shape(size_m, size_n, size_k);
  if (rc != VAQ_OK) return rc;
  VAQ_CHECK_ARG(dtype == VAQ_F16 || dtype == VAQ_BF16, "w4a16_gemm: only supports bfloat16 and float16 (dtype tag %d)",
                dtype);
  int wt = 0, sub = 1;
  bool channelwise = false;
  rc = check_format(size_k, group_size, wtype, &wt, &sub, &channelwise);
  if (rc != VAQ_OK) return rc;
  VAQ_CHECK_ARG((wtype == VAQ_WTYPE_U4) == (zeros != nullptr),
                "w4a16_gemm: b_q_type must be uint4 when has_zp = True and uint4b8, uint8b128 or float8_e4m3fn when has_zp = False");
  const bool w8 = wt != 0;
  VAQ_CHECK_SUPPORTED(wt != 2 || (sub == 1 && perm == nullptr),
                      "w4a16_gemm: FP8 weights take channelwise scales or groups of 128 rows, and no act_order");
  VAQ_CHECK_ARG(!w8 || size_k * size_n < (1ll << 32), "w4a16_gemm: problem too large for 8-bit weights");
  VAQ_CHECK_ARG(force_path >= 0 && force_path <= 2, "w4a16_gemm: force_path = %d", force_path);
  if (size_m == 0) return VAQ_OK;
  VAQ_CHECK_ARG(a && b && scales && c, "w4a16_gemm: null pointer");
  VAQ_CHECK_ARG(lda >= size_k && lda % 8 == 0, "w4a16_gemm: A.stride(0) = %lld must be >= size_k and divisible by 8",
                (long long)lda);
  VAQ_CHECK_ARG(((uintptr_t)a % 16) == 0, "w4a16_gemm: A must aligned to 16 bytes");
  VAQ_CHECK_ARG(((uintptr_t)b % 16) == 0 && ((uintptr_t)scales % 8) == 0 && ((uintptr_t)c % 8) == 0,
                "w4a16_gemm: b_q_weight must be 16-byte, b_scales and c 8-byte aligned");
  VAQ_CHECK_ARG(!perm || ((uintptr_t)perm % 16) == 0, "w4a16_gemm: perm must be 16-byte aligned");
  VAQ_CHECK_ARG(!bias || ((uintptr_t)bias % 8) == 0, "w4a16_gemm: bias must be 8-byte aligned");
  hipStream_t s = (hipStream_t)stream;

  if (perm && force_path == 0 && size_m * lda * 2 < (1ll << 31) && permutes_first((int)size_m, (int)size_n, (int)size_k, sub, w8)) {
    // into a_tmp beyond 32 rows, and into the end of c_tmp up to there, where what is left of it is enough for the call without act_order
    int64_t left = c_tmp_bytes;
    void* columns = a_tmp;
    if (size_m <= DECODE_MAX_M_2BLK) {
      left = (c_tmp_bytes - size_m * size_k * 2) & ~15ll;
      columns = c_tmp != nullptr && left >= 0 && small_call_fits((int)size_m, (int)size_n, (int)size_k, sub, wt, left, counters != nullptr ? counter_ints : 0)
                    ? reinterpret_cast<char*>(c_tmp) + left : nullptr;
    }
    if (columns != nullptr && ((uintptr_t)columns % 16) == 0) {
      rc = vaq_permute_cols(a, lda, perm, columns, size_m, size_k, stream);
      if (rc != VAQ_OK) return rc;
      rc = dispatch(columns, size_k, b, scales, zeros, nullptr, true, bias, c, left > 0 ? c_tmp : nullptr, left, a_tmp, counters, counter_ints, size_m, size_n,
                    size_k, sub, channelwise, wt, dtype, 0, s);
      if (rc != VAQ_ERR_INVALID_ARG) return rc;      // (beyond 32 rows, given too little scratch for that plan: as without it)
    }
  }
  return dispatch(a, lda, b, scales, zeros, perm, perm != nullptr, bias, c, c_tmp, c_tmp_bytes, a_tmp, counters, counter_ints, size_m, size_n, size_k,
                  sub, channelwise, wt, dtype, force_path, s);
}

// ----------------------------------------------------------------------------- the GEMM on library-owned scratch
namespace vaq {

// Scratch of vaq_w4a16_gemm_static: arrival counters (zero when the module is loaded, left zero by every kernel), then
// the split-K partial tiles, then the permuted activations.  One copy per GPU, held from the first use of the library
// on that GPU until the process ends.
constexpr size_t STATIC_COUNTER_INTS = VAQ_STATIC_SCRATCH_COUNTER_INTS;
constexpr size_t STATIC_DATA_BYTES = VAQ_STATIC_SCRATCH_DATA_BYTES;
static __device__ __align__(256) unsigned char scratch[STATIC_COUNTER_INTS * 4 + STATIC_DATA_BYTES];

// `scratch` above is the host-side handle of the array, not an address a kernel can use: the device address is looked up
// once per device, with that device current, and kept here.
static unsigned char* g_scratch_ptr[VAQ_MAX_DEVICES];
static hipError_t g_scratch_err[VAQ_MAX_DEVICES];
static std::once_flag g_scratch_once[VAQ_MAX_DEVICES];

static int static_scratch_of_current_device(unsigned char** out) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= VAQ_MAX_DEVICES) {
    (void)hipGetLastError();
    set_error("w4a16_gemm_static: cannot identify the current device");
    return VAQ_ERR_LAUNCH;
  }
  std::call_once(g_scratch_once[dev], [dev] {
    void* p = nullptr;
    g_scratch_err[dev] = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    g_scratch_ptr[dev] = g_scratch_err[dev] == hipSuccess ? static_cast<unsigned char*>(p) : nullptr;
    if (g_scratch_err[dev] != hipSuccess) (void)hipGetLastError();
  });
  if (g_scratch_ptr[dev] == nullptr) {
    set_error("w4a16_gemm_static: hipGetSymbolAddress failed on device %d: %s", dev, hipGetErrorString(g_scratch_err[dev]));
    return VAQ_ERR_LAUNCH;
  }
  *out = g_scratch_ptr[dev];
  return VAQ_OK;
}

}  // namespace vaq

extern "C" int vaq_w4a16_gemm_static(const void* a, int64_t lda, const int32_t* b, const void* scales,
                                     const int32_t* zeros, const int32_t* perm, const void* bias, void* c, int64_t size_m,
                                     int64_t size_n, int64_t size_k, int group_size, int dtype, int wtype, void* stream) {
  using namespace vaq;
  size_t c_tmp_bytes = 0, a_tmp_bytes = 0, counter_ints = 0;
  // The tile kernel's option of splitting the tiles of a half-empty last round over K is left out here: it is worth
  // tens of MB of partial tiles at thousands of rows, and whole tiles give the same result.
  VaqTuning whole_tiles = {};
  whole_tiles.exp[10] = 1;
  // What act_order's permuted activations leave of the scratch is what the K split may use for its partial tiles: a plan
  // that asked for more would have the call refused, where a smaller split, or none, gives the same result.
  const size_t perm_bytes = perm != nullptr && size_m > DECODE_MAX_M_2BLK && size_k > 0 ? (size_t)size_m * (size_t)size_k * 2 : 0;
  whole_tiles.exp[14] = perm_bytes + 1024 < STATIC_DATA_BYTES ? (int)((STATIC_DATA_BYTES - perm_bytes) / 1024) : 1;
  int rc = vaq_w4a16_gemm_workspace_tuned(size_m, size_n, size_k, perm != nullptr, 0, &c_tmp_bytes, &a_tmp_bytes, &counter_ints,
                                          &whole_tiles);
  if (rc != VAQ_OK) return rc;
  if (perm != nullptr && (counter_ints > STATIC_COUNTER_INTS || ((c_tmp_bytes + 255) & ~(size_t)255) + a_tmp_bytes > STATIC_DATA_BYTES)) {
    // the routes without the launch that permutes ahead of the decode kernels ask for less
    whole_tiles.exp[9] = 1;
    rc = vaq_w4a16_gemm_workspace_tuned(size_m, size_n, size_k, 1, 0, &c_tmp_bytes, &a_tmp_bytes, &counter_ints, &whole_tiles);
    if (rc != VAQ_OK) return rc;
  }
  const size_t c_tmp_span = (c_tmp_bytes + 255) & ~(size_t)255;
  VAQ_CHECK_ARG(counter_ints <= STATIC_COUNTER_INTS && c_tmp_span + a_tmp_bytes <= STATIC_DATA_BYTES,
                "w4a16_gemm_static: M=%lld N=%lld K=%lld needs %zu counters and %zu + %zu bytes of scratch, the "
                "library-owned scratch holds %zu counters and %zu bytes; use vaq_w4a16_gemm with caller scratch",
                (long long)size_m, (long long)size_n, (long long)size_k, counter_ints, c_tmp_bytes, a_tmp_bytes,
                STATIC_COUNTER_INTS, STATIC_DATA_BYTES);
  unsigned char* base = nullptr;
  if (size_m > 0) {
    rc = static_scratch_of_current_device(&base);
    if (rc != VAQ_OK) return rc;
  }
  int32_t* counters = reinterpret_cast<int32_t*>(base);
  unsigned char* data = base ? base + STATIC_COUNTER_INTS * 4 : nullptr;
  return vaq_w4a16_gemm_tuned(a, lda, b, scales, zeros, perm, bias, c, c_tmp_bytes ? reinterpret_cast<float*>(data) : nullptr,
                              (int64_t)c_tmp_bytes, a_tmp_bytes ? data + c_tmp_span : nullptr, counters,
                              (int64_t)STATIC_COUNTER_INTS, size_m, size_n, size_k, group_size, dtype, wtype, 0, stream,
                              &whole_tiles);
}
