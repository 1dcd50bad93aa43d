// Host side of the LDS-staged decode kernel (w4a16_decode2_kernel.h): configuration choice, workspace sizes, launch
// of the instances for quantisation groups of 128 rows and channelwise scales.
#include "tile_plan.h"
#include "w4a16_decode2_kernel.h"
#include "w4a16_kernels.h"

namespace vaq {

// ----------------------------------------------------------------------------- host side

struct Decode2Config {
  int gs, wks, wn, sk, mr;
  int rc;      // ring variant of long streams (see the kernel): 0 two slots refilled early, 1 / 2 four / three slots refilled late
};

static inline bool exp_off(const VaqTuning& tn, int i) { return tn.exp[i] != 1; }      // development switch i not set to "off"

static int round_gs(int x, int sub, bool w8) {
  const int opts[] = {1, 2, 4, 7, 8, 14, 16};
  for (int o : opts) {
    if (sub > 1 && (o & (o - 1)) != 0) continue;     // sub-group instances exist for powers of two only
    if (w8 && (o & 1)) continue;                     // 8-bit codes: two tiles (nibble planes) per group
    if (o >= x) return o;
  }
  return 16;
}

// Workgroups of `waves` wavefronts and `lds_wg` bytes of LDS that share a compute unit (at least one).
static inline long wg_slots(int waves, size_t lds_wg) {
  const long by_waves = D2_WAVES / waves, by_lds = (long)((size_t)(160 * 1024) / lds_wg);
  const long slots = by_waves < by_lds ? by_waves : by_lds;
  return slots < 1 ? 1 : slots;
}

// n-tiles per workgroup (at most 16 / wks).  A compute unit holds 16 of these wavefronts and as many workgroups as its LDS
// allows (`lds_wg` bytes each).  First the fewest rounds of workgroups per compute unit, then the fewest wavefronts on the
// busiest compute unit (i.e. spread over the device), then the smaller workgroup.
static int pick_wn(int NT, int sk, int wks, size_t lds_wg, long* rounds_out) {
  const int cus = num_cus_current_device();
  int best_wn = 1;
  long best_rounds = -1, best_waves = -1;
  for (int wn = 1; wn <= D2_WAVES / wks; ++wn) {
    const long slots = wg_slots(wks * wn, lds_wg);
    const long wgs = (long)((NT + wn - 1) / wn) * sk;
    const long per_cu = (wgs + cus - 1) / cus;
    const long rounds = (per_cu + slots - 1) / slots;
    const long waves = (per_cu < slots ? per_cu : slots) * wn * wks;
    if (best_rounds < 0 || rounds < best_rounds || (rounds == best_rounds && waves < best_waves)) {
      best_rounds = rounds;
      best_waves = waves;
      best_wn = wn;
    }
  }
  if (rounds_out) *rounds_out = best_rounds;
  return best_wn;
}

// Groups per slab are limited by LDS (128 KiB of activations, 256 bytes per group and staged row): 512 / rows.
// G, gslab, gs and slab_max below count weight tiles: one per 128 rows of K, two (nibble planes) for 8-bit codes.
// `nt_mult`: copies of every n-tile's stream that run side by side (rows split over workgroups, see the kernel).
static Decode2Config pick_by_rule(int M, int N, int K, int sub, bool w8, int nt_mult = 1, bool allow8 = true) {
  const int TPG = w8 ? 2 : 1;
  const int G = K / 128 * TPG, NT = N / 16 * nt_mult;
  const int MB = (M + 15) / 16;
  Decode2Config c;
  c.mr = M == 1 ? 1 : (M <= 4 ? 4 : (M <= 8 && sub == 1 && !w8 && allow8 && tuning().exp[3] != 1 ? 8 : 16));      // rows staged (8: 4-bit codes in groups of 128 rows only)
  const int slab_max = 512 / (c.mr * MB) * TPG;
  c.sk = (G + slab_max - 1) / slab_max;
  const int gslab = (G + c.sk - 1) / c.sk;            // groups per slab
  const int cus = num_cus_current_device();
  // K slices wanted: about 16 wavefronts per compute unit, 8 when few rows are staged (measured: with little LDS to
  // fill, longer per-wavefront tile streams beat more wavefronts on layers with few n-tiles)
  // (also with 16 staged rows when there is at most one workgroup per compute unit: 4096 x 4096 at M = 16, 6.60 -> 6.34 us)
  // (and with 16 staged rows on up to two (n-tile, K slab) pairs per compute unit: four K slices of 8 tiles with the
  // three-slot ring below, 4096 x 6144 at M = 16 6.9 -> 6.5 us, 8192 x 6144 10.9 -> 9.5 us, 4096 x 8192 7.5 -> 7.0 us)
  int want = (cus * ((NT * c.sk <= 2 * cus && MB == 1) || NT * c.sk <= cus ? 8 : D2_WAVES)) / (NT * c.sk);
  int wks = 1;
  while (wks * 2 <= want && wks < 16) wks *= 2;
  while (wks > 1 && wks > gslab) wks /= 2;
  // A single row: as many K slices as it takes to cover K with streams of at most 16 tiles, rather than a split over
  // workgroups and its hand-over (28672 x 8192 at M = 1: 30.2 -> 24.5 us, 28672 x 4096 17.7 -> 14.8 us; from two rows on
  // the split wins or ties) -- where those workgroups, one per n-tile, make full rounds (20480 x 5120, 320 n-tiles:
  // 16.7 -> 19.4 us).
  if (c.mr == 1 && (NT <= cus || NT % cus == 0 || (NT % cus) * 5 >= cus * 4))
    while (wks < 16 && wks * 16 < gslab) wks *= 2;
  const VaqTuning& tn = tuning();
  // Two m-blocks of a long K on a layer of at most one n-tile per compute unit: slabs of one 14-tile stream per
  // wavefront with the four-slot ring (14336 x 4096 at M = 17 / 32: 13.8 / 14.7 -> 12.9 / 13.2 us; 11008 x 4096 14.1 -> 12.4 us;
  // 16-tile streams, two slices of 7 or 8, and the same on 8192 x 8192 or a 28672-wide layer are slower).
  bool long_k_two_blocks = MB == 2 && NT <= cus && G >= 80 && sub == 1 && !w8 && nt_mult == 1;
  if (long_k_two_blocks) {
    // ... and only as one round of workgroups of 7 to 10 wavefronts that fill 85 % of the device (measured slower with
    // 4, 11 and 15 wavefronts: 14336 x 2048 10.3 -> 12.2 us, 16384 x 4096 14.2 -> 15.5 us, 24576 x 4096 18.9 -> 20.3 us)
    const int sk_b = (G + 13) / 14;
    long rounds_b = 0;
    const int wn_b = pick_wn(NT, sk_b, 1, decode2_lds_bytes(1, 14, c.mr, MB), &rounds_b);
    const long wgs_b = (long)((NT + wn_b - 1) / wn_b) * sk_b;
    long_k_two_blocks = rounds_b == 1 && wn_b >= 7 && wn_b <= 10 && wgs_b * 100 >= (long)cus * 85;
  }
  if (long_k_two_blocks) wks = 1;
  if (tn.decode2_wks > 0) wks = tn.decode2_wks;
  int gs = long_k_two_blocks ? 14 : round_gs((gslab + wks - 1) / wks, sub, w8);
  if (tn.decode2_gs > 0) gs = tn.decode2_gs;
  while (wks * gs > slab_max && wks > 1) wks /= 2;     // respect the LDS limit
  if (gs > slab_max) {                                 // rounding up went past it: largest instantiated size below
    const int opts[] = {8, 7, 4, 2, 1};
    for (int o : opts)
      if (o <= slab_max && !(w8 && (o & 1)) && !(sub > 1 && (o & (o - 1)) != 0)) {
        gs = o;
        break;
      }
  }
  // Two slabs that twice the K slices would cover as one (at most 15 % of their tiles beyond K): one slab, no hand-over
  // between workgroups.  Cold, M = 1 / 4 / 16: 3584 x 37888 (16 + 12 groups) 20.3 / 27.8 / 23.2 -> 17.7 / 17.7 / 19.6 us,
  // 13824 x 5120 (64 + 44) 12.1 / 12.9 -> 11.0 / 11.9 us.
  if (MB == 1 && sub == 1 && !w8 && !long_k_two_blocks && tn.decode2_gs <= 0 && tn.decode2_wks <= 0 && exp_off(tn, 5) &&
      (G + wks * gs - 1) / (wks * gs) == 2 && wks * 2 <= 16) {
    const int g2 = round_gs((G + 2 * wks - 1) / (2 * wks), sub, w8);
    const int cover = 2 * wks * g2;
    if (cover >= G && cover <= slab_max && (cover - G) * 100 <= G * 15) {
      wks *= 2;
      gs = g2;
    }
  }
  // A last slab of less than 35 % of the others on a layer of at most two n-tiles per compute unit: the stream length
  // (same K slices) that leaves the fewest tiles beyond K, a further slab counted as 3 %.  Cold, M = 1 / 4: 9216 x 4608
  // (64 + 8 groups -> 3 x 28) 11.0 / 12.1 -> 8.9 / 9.3 us, 18944 x 3584 at M = 4 (64 + 64 + 20 -> 3 x 56) 13.5 -> 12.0 us; on
  // a wide layer the further slab costs more than it brings (5120 x 27648, 32 + 8 -> 3 x 14: +3 .. +13 %).
  if (MB == 1 && sub == 1 && !w8 && !long_k_two_blocks && tn.decode2_gs <= 0 && tn.decode2_wks <= 0 && exp_off(tn, 5) &&
      NT <= 2 * cus) {
    auto slabs = [&](int g) { return (G + wks * g - 1) / (wks * g); };
    const int sk0 = slabs(gs), last = G - (sk0 - 1) * wks * gs;
    if (sk0 >= 2 && last * 20 < wks * gs * 7) {
      auto score = [&](int g) { return (double)(slabs(g) * wks * g - G) / G + 0.03 * slabs(g); };
      int bg = gs;
      double best = score(gs);
      for (int g : {16, 14, 8, 7}) {
        if (wks * g > slab_max || slabs(g) > 10) continue;
        if (score(g) < best - 1e-9) { best = score(g); bg = g; }
      }
      gs = bg;
    }
  }
  // One slab whose streams reach 35 % and more beyond K (wavefronts without tiles) on a layer of at most 1.25 n-tiles per
  // compute unit: two or three slabs of streams of 7 tiles and more (the K slices as planned or half of them) that fit K
  // better.  Cold, M = 2 / 4 / 16: 5120 x 5120 (4 x 14 for 40 groups -> 3 slabs of 2 x 7) 7.9 / 7.9 / 8.6 -> 6.9 / 6.9 / 7.4 us,
  // 10240 x 2560 (8 x 14 for 80 -> 3 slabs of 4 x 7) 8.0 / 8.0 -> 6.8 / 6.9 us, 9216 x 2304 8.0 -> 6.8 us; wider layers lose with
  // it (2560 x 10240, 5120 x 15360: +20 .. +60 %), so do a single row (10240 x 4096: +18 %) and a K of 2560 (+11 .. +14 %);
  // 10240 x 4096 at M = 2 / 4 is 3 % slower with it.
  if (MB == 1 && sub == 1 && !w8 && !long_k_two_blocks && tn.decode2_gs <= 0 && tn.decode2_wks <= 0 && exp_off(tn, 5) &&
      c.mr >= 4 && G >= 32 && NT * 4 <= cus * 5 && wks <= 8 && wks * gs >= G && (wks * gs - G) * 100 >= G * 35) {
    auto slabs = [&](int w, int g) { return (G + w * g - 1) / (w * g); };
    auto score = [&](int w, int g) { return (double)(slabs(w, g) * w * g - G) / G + 0.03 * slabs(w, g); };
    int bw = wks, bg = gs;
    double best = score(wks, gs);
    for (int w : {wks, wks / 2}) {
      if (w < 1) continue;
      for (int g : {14, 8, 7}) {
        if (w * g > slab_max || slabs(w, g) > 3) continue;
        if (score(w, g) < best - 1e-9) { best = score(w, g); bw = w; bg = g; }
      }
    }
    wks = bw;
    gs = bg;
  }
  // the slab is now wks*gs groups; recompute the number of slabs
  c.sk = (G + wks * gs - 1) / (wks * gs);
  c.gs = gs;
  c.wks = wks;
  const size_t lds_wg = decode2_lds_bytes(wks, gs / TPG, c.mr, MB);
  const int best_wn = pick_wn(NT, c.sk, wks, lds_wg, nullptr);
  c.wn = tn.decode2_wn > 0 ? tn.decode2_wn : best_wn;
  if (c.wn * wks > D2_WAVES) c.wn = D2_WAVES / wks;
  // ring variant of long streams (instances exist for 4-bit codes in groups of 128 rows / channelwise, up to two
  // m-blocks): by the wavefronts that share a compute unit
  c.rc = 0;
  if (sub == 1 && !w8 && MB <= 2 && gs >= 7) {
    const long slots = wg_slots(wks * c.wn, lds_wg);
    const long per_cu = ((long)((NT + c.wn - 1) / c.wn) * c.sk + cus - 1) / cus;
    const long waves_cu = (per_cu < slots ? per_cu : slots) * wks * c.wn;
    if (long_k_two_blocks && wks == 1 && gs == 14) c.rc = 1;
    else if (c.mr >= 8 && (gs >= 8 || waves_cu <= 8)) c.rc = 2;      // (7 tiles per wavefront, 16 wavefronts, 14336 x 4096 at M = 16: three slots 11.5 us, two 11.2 us)
    else if (waves_cu <= 8) c.rc = 1;
  }
  if (tn.exp[1] > 0) c.rc = tn.exp[1] - 1;      // (development switch: forced ring variant + 1)
  // 8 staged rows allow slabs twice as long, and a slab is a whole number of instantiated stream lengths: where that
  // leaves a last slab of less than 60 % of the others the workgroups of the full slabs set the pace, and the plan for
  // 16 staged rows (shorter, evener slabs) is taken instead (M = 8, cold: 10240 x 2560, slabs of 56 + 24 groups, 9.7 us
  // against 7.5 us; 5120 x 27648, 32 + 8, 23.2 against 20.8 us; 17920 x 6656, 4 x 32 + 12, 20.0 against 16.9 us)
  if (c.mr == 8 && c.sk > 1 && tn.decode2_gs <= 0 && tn.decode2_wks <= 0) {
    const int slab = c.wks * c.gs, last = G - (c.sk - 1) * slab;
    if (last * 10 < slab * 6) return pick_by_rule(M, N, K, sub, w8, nt_mult, false);
  }
  return c;
}

// ----------------------------------------------------------------------------- plans by predicted time
// What a launch costs, in us: per round of workgroups on a compute unit `round` over the workgroups that share it, the activation
// fill (`fill_kb` per KB staged on it), the stream of weight tiles -- per tile `chain` and the latency `tile_latency` over the
// tiles in flight, or the arithmetic of all wavefronts that share the unit, `tile_work` each -- and the reduction over the K
// slices (`reduce` per doubling); a started round beyond the first counts by `last` beyond its share; workgroups of two
// wavefronts, more than four to a unit, take `pair` times as long; beside that the weights from memory (`mem_mb` per MB, and
// `again` times that for every further copy of the stream, which L2 serves); `base` per launch; a K split over workgroups costs
// `handover` + `part` per part + `part_mb` per MB of partial results.  [.]: one staged row, 4 or 8, 16.  `sub_work`: groups of
// 128, 64, 32 rows.  `spread`: rows over workgroups, the copies of an n-tile range are a grid row (gx workgroups) apart and meet on
// one XCD only if 8 divides gx; with gx odd they are on all eight, each of which brings the stream into its L2 (14-20 % of a launch
// below 4 MB of weights, 6-10 % to 16 MB: 1 .. 1.5 us whatever the size).  768 x 704 at M = 201 5.6 -> 4.2 us (one n-tile to a
// workgroup, gx = 44, instead of three, gx = 15), 1792 x 8192 at M = 98 14.4 -> 12.3 us; over 6808 problems whose plan it changes
// 3.3 % in the mean.
// Fitted to the cold times of 1.5e5 launches: 6400 problems of random layers, half of them with K 1024 .. 14336 and N 1024 ..
// 28672, half with K 256 .. 28672 and N 256 .. 152064, 1 .. 256 rows, each with up to 60 splits (the first part of those in
// profiles/plan_prices; rows over workgroups with 8-bit codes and `spread` to all of them).  The cheapest plan by these figures takes
// 1.016 of the fastest one's time (geometric mean over 16672 problems; 99 of 100 less than 1.21), N > 28672 1.026, K or N below 1024
// 1.013.  Constants of the formula without `chain`, `last` and `pair`, fitted to the first half only, were at 1.047, 1.067
// and 1.060 over these problems.
struct Decode2Cost {
  double base, round, fill_kb, mem_mb, again, reduce, handover, part, part_mb;
  double tile_latency[3], tile_work[3], sub_work[3];
  double chain, last, pair, spread;
};
constexpr Decode2Cost D2_COST_W8 = {1.09, 1.63, 0.0154, 0.0469, 0, 0.00669, 1.12, 0.275, 0.409,
                                    {0.9, 0.875, 0.665}, {0.0215, 0.022, 0.0209}, {1.15, 1.35, 1.95}, 0.116, 0.108, 1.29, 0};
constexpr Decode2Cost D2_COST_SUB = {1.18, 1.3, 0.0144, 0.0468, 0, 0.0041, 1.16, 0.301, 0,
                                     {0.796, 0.909, 0.834}, {0.0278, 0.0271, 0.028}, {1, 1.11, 1.55}, 0.127, 0.143, 1.35, 0};
// two m-blocks (groups of 128 rows / channelwise: three and four)
constexpr Decode2Cost D2_COST_W8_MB2 = {0.149, 0.0523, 0.000908, 0.0746, 0, 0.848, 0.588, 0.231, 0.597,
                                        {1.8, 1.8, 1.59}, {0.0586, 0.0586, 0.0342}, {1.41, 1.65, 2.41}, 0.142, 0.428, 1.06, 0};
constexpr Decode2Cost D2_COST_SUB_MB2 = {0.772, 0.979, 0.0147, 0.071, 0, 0.218, 0.395, 0.3, 0.46,
                                         {1.84, 1.84, 1.63}, {0.0643, 0.0643, 0.0498}, {1, 1.08, 1.46}, 0.0313, 0.379, 0.968, 0};
constexpr Decode2Cost D2_COST_MB34 = {1.97, 1.26, 0.0179, 0.158, 0, 0.0465, 0.224, 0.328, 0.782,
                                      {1.97, 1.97, 0.468}, {0.0886, 0.0886, 0.00497}, {1.72, 1, 1}, 0.107, 0.395, 1.2, 0};
// 4-bit codes in groups of 128 rows / channelwise by up to 16 rows, whose plan is the rule's: to weigh that against the kernel with activations in
// registers (up to 4 and 5 .. 16 rows; two m-blocks; 2600 problems of profiles/plan_prices, 5-6 % rms)
constexpr Decode2Cost D2_COST_4 = {2.27, 0.561, 0.00957, 0.196, 0, 0.000523, 1.17, 0.118, 0.0294,
                                   {0.0249, 0.0232, 0.834}, {0.0315, 0.0343, 0.028}, {0.93, 1.11, 1.55}, 0.0824, 0.594, 1.15, 0};
constexpr Decode2Cost D2_COST_16 = {2.34, 0.579, 0.0093, 0.185, 0, 0.00117, 0.907, 0.198, 0.305,
                                    {0.796, 0.0366, 0.215}, {0.0278, 0.107, 0.105}, {0.372, 1.11, 1.55}, 0.00252, 0.143, 1.36, 0};
constexpr Decode2Cost D2_COST_MB2 = {2.74, 0.146, 0.0153, 0.13, 0, 0.00417, 0.659, 0.209, 0.283,
                                     {1.84, 1.84, 0.0436}, {0.0643, 0.0643, 0.0314}, {1.55, 1.08, 1.46}, 0.0769, 0.379, 0.864, 0};
// the rows split over workgroups (never with a split K)
constexpr Decode2Cost D2_COST_ROWS_W8 = {1.15, 1.41, 0.013, 0.409, 0.0868, 0.0134, 0, 0, 0,
                                         {0.86, 0.86, 0.411}, {0.0336, 0.0336, 0.0173}, {1.27, 1.51, 2.19}, 0.113, 0.146, 1.2, 2.57};
constexpr Decode2Cost D2_COST_ROWS_SUB = {1.54, 1.24, 0.0103, 0.229, 0.267, 0.00948, 0, 0, 0,
                                          {1.36, 1.36, 0.0918}, {0.0476, 0.0476, 0.0195}, {1, 1.49, 2.01}, 0.151, 0.153, 1.2, 1.5};
constexpr Decode2Cost D2_COST_ROWS = {1.4, 1.16, 0.0093, 0.0946, 0.368, 0.0106, 0, 0, 0,
                                      {1.02, 1.02, 0.392}, {0.037, 0.037, 0.0181}, {1.74, 1, 1}, 0.107, 0.237, 1.2, 1.5};

static const Decode2Cost& workgroup_cost(int M, int sub, bool w8) {
  if (w8) return M > 16 ? D2_COST_W8_MB2 : D2_COST_W8;
  if (sub > 1) return M > 16 ? D2_COST_SUB_MB2 : D2_COST_SUB;
  return M > 32 ? D2_COST_MB34 : M > 16 ? D2_COST_MB2 : M > 4 ? D2_COST_16 : D2_COST_4;
}

static double decode2_us(const Decode2Cost& t, const Decode2Config& c, int M, int N, int K, int sub, bool w8, int MB, int copies) {
  const int cus = num_cus_current_device(), TPG = w8 ? 2 : 1;
  const int ri = c.mr == 1 ? 0 : c.mr <= 8 ? 1 : 2;
  const long slots = wg_slots(c.wks * c.wn, decode2_lds_bytes(c.wks, c.gs / TPG, c.mr, MB));
  const long wgs = (long)((N / 16 + c.wn - 1) / c.wn) * c.sk * copies, per_cu = (wgs + cus - 1) / cus;
  const double side = (double)(per_cu < slots ? per_cu : slots), even = (double)per_cu / (double)slots;
  const double rounds = per_cu > slots ? even + t.last * ((double)((per_cu + slots - 1) / slots) - even) : 1;
  const bool whole = c.mr <= 4 && c.gs <= (sub > 1 ? 4 : 8);      // short streams with few rows are requested whole
  const double flight = whole || c.gs < 3 ? c.gs : 3;
  auto p4 = [](double x) { return x * x * x * x; };
  const double tile = sqrt(sqrt(p4(t.tile_latency[ri] / flight) +
                                p4(side * c.wks * c.wn * t.tile_work[ri] * t.sub_work[sub == 4 ? 2 : sub - 1]))) +
                      t.chain * t.sub_work[sub == 4 ? 2 : sub - 1];
  const double fill = t.fill_kb * side * (c.wks * c.gs / TPG) * (c.mr * MB * 256 / 1024.0);
  const double slow = c.wks * c.wn == 2 && per_cu > 4 ? t.pair : 1;
  const double core = slow * rounds * (t.round / (double)slots + fill + c.gs * tile + t.reduce * log2((double)c.wks));
  const double mem = t.mem_mb * 0.5e-6 * (double)K * N * TPG * (1 + t.again * (copies - 1));
  double us = t.base + cbrt(core * core * core + mem * mem * mem);
  if (c.sk > 1) us += t.handover + c.sk * (t.part + t.part_mb * 4e-6 * (double)M * N);
  if (copies > 1) {
    const long gx = (N / 16 + c.wn - 1) / c.wn, xcds = gx % 8 == 0 ? 1 : gx % 4 == 0 ? 2 : gx % 2 == 0 ? 4 : 8;
    us += t.spread * (double)((copies < xcds ? copies : xcds) - 1) / 7.0;
  }
  return us;
}

struct Decode2Plan {
  Decode2Config c{};
  double us = -1;      // predicted; negative: no plan
};

// The cheapest plan of one workgroup for all rows (rows == false) or of workgroups of 16 rows each.
static Decode2Plan cheapest_decode2(const Decode2Cost& t, int M, int N, int K, int sub, bool w8, bool rows) {
  const int TPG = w8 ? 2 : 1, G = K / 128 * TPG, NT = N / 16;
  const int copies = rows ? (M + 15) / 16 : 1, MB = rows ? 1 : (M + 15) / 16;
  const VaqTuning& tn = tuning();
  Decode2Plan best;
  Decode2Config c{};
  c.mr = rows ? 16 : M == 1 ? 1 : M <= 4 ? 4 : 16;
  const int slab_max = 512 / (c.mr * MB) * TPG;
  for (int gs : {1, 2, 4, 7, 8, 14, 16}) {
    if (gs != round_gs(gs, sub, w8)) continue;
    if (tn.decode2_gs > 0 && gs != tn.decode2_gs) continue;
    for (int wks = 1; wks <= 16; wks *= 2) {
      if (tn.decode2_wks > 0 && wks != tn.decode2_wks) continue;
      // (four sub-grouped tiles of two m-blocks, unrolled whole, do not fit the registers: twice the time of eight)
      if (MB == 2 && sub == 4 && gs == 4 && !w8 && tn.decode2_gs <= 0) continue;
      if (wks * gs > slab_max || (wks > 1 && gs > 2 && wks * gs >= 2 * G)) continue;
      c.gs = gs;
      c.wks = wks;
      c.sk = (G + wks * gs - 1) / (wks * gs);
      if (rows && c.sk != 1) continue;
      if (c.sk > 8 && tn.decode2_gs <= 0) continue;
      if (c.sk > 1 && K <= 2048 && tn.decode2_gs <= 0) continue;       // (fits one slab whatever the format: no hand-over)
      if (c.sk > 1 && (size_t)c.sk * NT * MB * 1024 > VAQ_STATIC_SCRATCH_DATA_BYTES) continue;      // (the library-owned scratch)
      const int fixed = tn.decode2_wn > 0 ? min(tn.decode2_wn, D2_WAVES / wks)
                                          : rows ? 0 : pick_wn(NT, c.sk, wks, decode2_lds_bytes(wks, gs / TPG, c.mr, MB), nullptr);
      for (int wn = fixed > 0 ? fixed : 1; wn <= (fixed > 0 ? fixed : D2_WAVES / wks); ++wn) {
        if (fixed <= 0 && wks * wn < 4) continue;
        c.wn = wn;
        const double us = decode2_us(t, c, M, N, K, sub, w8, MB, copies);
        if (best.us >= 0 && us >= best.us) continue;
        best.us = us;
        best.c = c;
      }
    }
  }
  if (rows && best.us >= 0 && sub == 1 && !w8 && best.c.gs >= 7) {      // the ring, as in pick_by_rule
    const int cus = num_cus_current_device();
    const long slots = wg_slots(best.c.wks * best.c.wn, decode2_lds_bytes(best.c.wks, best.c.gs, 16, 1));
    const long per_cu = ((long)((NT + best.c.wn - 1) / best.c.wn) * copies + cus - 1) / cus;
    if (best.c.gs >= 8 || (per_cu < slots ? per_cu : slots) * best.c.wks * best.c.wn <= 8) best.c.rc = 2;
    if (tn.exp[1] > 0) best.c.rc = tn.exp[1] - 1;
  }
  return best;
}

// One workgroup for all rows (up to two m-blocks; 4-bit codes in groups of 128 rows / channelwise: up to four).  The rule for the
// latter, whose choices are within 2-4 % of the predicted ones up to two m-blocks.  For the other formats, which the rule was not
// made for, the cheapest plan where it is predicted 5 % (4-bit codes in groups of 64 / 32 rows, up to 16 rows: 8 %) ahead of the
// rule's: nearer than that the price is more often wrong than right (over 3863 problems the mean gain over the rule is 4.7-10.4 %
// either way, the share that is 5 % slower than by the rule falls from 3-8 % to 1-3 %).
static Decode2Plan plan_workgroup(int M, int N, int K, int sub, bool w8) {
  Decode2Plan p;
  p.c = pick_by_rule(M, N, K, sub, w8);
  p.us = decode2_us(workgroup_cost(M, sub, w8), p.c, M, N, K, sub, w8, (M + 15) / 16, 1);
  if (sub > 1 || w8) {
    const Decode2Plan q = cheapest_decode2(workgroup_cost(M, sub, w8), M, N, K, sub, w8, false);
    const double ahead = w8 || M > 16 ? 0.95 : 0.92;
    if (q.us >= 0 && q.us < ahead * p.us) return q;
  }
  return p;
}

// Rows split over workgroups, one m-block each (see the kernel): needs no split of K.
static Decode2Plan plan_rows(int M, int N, int K, int sub, bool w8) {
  if (sub == 1 && !w8 && M <= 32) {      // by the rule, see w4a16_decode2_choose
    Decode2Plan p;
    p.c = pick_by_rule(16, N, K, sub, w8, (M + 15) / 16);
    p.us = decode2_us(D2_COST_ROWS, p.c, M, N, K, sub, w8, 1, (M + 15) / 16);
    if (p.c.sk == 1) return p;
  }
  return cheapest_decode2(w8 ? D2_COST_ROWS_W8 : sub > 1 ? D2_COST_ROWS_SUB : D2_COST_ROWS, M, N, K, sub, w8, true);
}

// Finished plans, one table per thread (see PlanTable); calls with this kernel's switches set neither read nor fill it.
template <class Make>
static Decode2Plan cached_plan(bool rows, int M, int N, int K, int sub, bool w8, Make make) {
  static thread_local PlanTable<Decode2Plan> table;
  const VaqTuning& tn = tuning();
  if (tn.decode2_gs > 0 || tn.decode2_wks > 0 || tn.decode2_wn > 0 || tn.exp[1] > 0 || tn.exp[3] > 0 || tn.exp[5] > 0) return make();
  return table.get(M, N, K, ((num_cus_current_device() * 8 + sub) * 2 + (w8 ? 1 : 0)) * 2 + (rows ? 1 : 0), make);
}
static Decode2Plan workgroup_plan(int M, int N, int K, int sub, bool w8) {
  return cached_plan(false, M, N, K, sub, w8, [&] { return plan_workgroup(M, N, K, sub, w8); });
}
static Decode2Plan rows_plan(int M, int N, int K, int sub, bool w8) {
  return cached_plan(true, M, N, K, sub, w8, [&] { return plan_rows(M, N, K, sub, w8); });
}

template <bool BF16, int MB, bool HAS_ZP, int MR, int GS>
static int dispatch_rc2(const Decode2Params& p, int rc, hipStream_t s) {
  if (rc == 1) return launch_decode2<BF16, GS, MB, HAS_ZP, MR, 1, 0, 1>(p, s);
  if (rc == 2) return launch_decode2<BF16, GS, MB, HAS_ZP, MR, 1, 0, 2>(p, s);
  if (rc == 3) return launch_decode2<BF16, GS, MB, HAS_ZP, MR, 1, 0, 3>(p, s);
  return launch_decode2<BF16, GS, MB, HAS_ZP, MR, 1>(p, s);
}

template <bool BF16, int MB, bool HAS_ZP, int MR>
static int dispatch_gs2(const Decode2Params& p, int gs, int rc, hipStream_t s) {
  switch (gs) {
    case 1: return launch_decode2<BF16, 1, MB, HAS_ZP, MR, 1>(p, s);
    case 2: return launch_decode2<BF16, 2, MB, HAS_ZP, MR, 1>(p, s);
    case 4: return launch_decode2<BF16, 4, MB, HAS_ZP, MR, 1>(p, s);
    case 7: return dispatch_rc2<BF16, MB, HAS_ZP, MR, 7>(p, rc, s);
    case 8: return dispatch_rc2<BF16, MB, HAS_ZP, MR, 8>(p, rc, s);
    case 14: return dispatch_rc2<BF16, MB, HAS_ZP, MR, 14>(p, rc, s);
    case 16: return dispatch_rc2<BF16, MB, HAS_ZP, MR, 16>(p, rc, s);
    default: break;
  }
  set_error("w4a16_gemm(decode): unsupported groups per wavefront %d", gs);
  return VAQ_ERR_UNSUPPORTED;
}

template <int MB, int MR>
static int dispatch_types2(const Decode2Params& p, int gs, int rc, bool bf16, bool zp, hipStream_t s) {
  if (bf16) return zp ? dispatch_gs2<true, MB, true, MR>(p, gs, rc, s) : dispatch_gs2<true, MB, false, MR>(p, gs, rc, s);
  return zp ? dispatch_gs2<false, MB, true, MR>(p, gs, rc, s) : dispatch_gs2<false, MB, false, MR>(p, gs, rc, s);
}

template <int MB>
static int dispatch_mr2(const Decode2Params& p, const Decode2Config& c, bool bf16, bool zp, hipStream_t s) {
  switch (c.mr) {
    case 1: return dispatch_types2<MB, 1>(p, c.gs, c.rc, bf16, zp, s);
    case 4: return dispatch_types2<MB, 4>(p, c.gs, c.rc, bf16, zp, s);
    case 8:
      if constexpr (MB == 1) return dispatch_types2<MB, 8>(p, c.gs, c.rc, bf16, zp, s);
      [[fallthrough]];
    default: return dispatch_types2<MB, 16>(p, c.gs, c.rc, bf16, zp, s);
  }
}

// Which kernel takes more than 16 rows: workgroups of all rows (`wg_ok`: built for this case), of 16 rows each, or the tile
// kernel (`tile_ok`, predicted to take `tile_us`).  No act_order inside (`has_perm`) and no FP8 weights among the workgroups of 16 rows.
// 17 .. 32 rows of 4-bit codes in groups of 128 rows / channelwise: 16 rows each where one m-block needs no split of K and one
// round of workgroups of at least eight wavefronts takes them all; 4096 x 4096 at M = 32 8.5 -> 6.3 us; a 28672-wide layer would
// need streams of 32 tiles (20.4 -> 21.7 us).  Everything else by predicted time.
// (development switch exp[2]: 1 never 16 rows each, 2 wherever it is built)
int w4a16_decode2_choose(int M, int N, int K, int sub, int wt, bool act_order, bool has_perm, bool wg_ok, bool tile_ok, double tile_us) {
  const bool w8 = wt != 0, rows_ok = M > 16 && M <= DECODE2_MAX_M_ROWS && wt != 2 && !has_perm && tuning().exp[2] != 1;
  if (!rows_ok && !tile_ok) return D2_WORKGROUP;
  Decode2Plan r;
  if (rows_ok) r = rows_plan(M, N, K, sub, w8);
  if (r.us >= 0 && tuning().exp[2] == 2) return D2_ROWS;
  if (wg_ok && M <= 32 && sub == 1 && !w8) {
    const long wgs = r.us >= 0 ? (long)((N / 16 + r.c.wn - 1) / r.c.wn) * ((M + 15) / 16) : 0;
    return r.us >= 0 && wgs <= num_cus_current_device() && r.c.wks * r.c.wn >= 8 ? D2_ROWS : D2_WORKGROUP;
  }
  int best = D2_TILE;
  // (`tile_us` is the price of the tile shapes with weights through LDS, see w4a16_staged_us, of 4-bit codes: 2-5 % low at these sizes,
  // 9-13 % with 8-bit codes; the prices of these workgroups are 3-9 % low.  With these factors the kind chosen is, against those shapes,
  // within 0.2 - 0.6 % of the fastest one's time in the mean, 1.3 % for groups of 64 / 32 rows at 17 .. 32 rows; 6600 problems.  The strips
  // that run in their place are up to 40 % faster; they take no problem from here because they round the scaled weights to 16 bits.
  // act_order: workgroups of all rows, with float32 scales, keep what they were given when the columns were always gathered inside them
  // and the tile kernel's launch for it was priced at 4 us; workgroups of 16 rows take calls from those only: the tile kernel gives the weights'
  // infinities where an activation is infinite, and finite results of huge ones, the decode kernel NaN.)
  double us = tile_ok ? tile_us * (!w8 ? 1.04 : M <= 64 ? 1.06 : 1.0) : -1;
  if (wg_ok) {
    const double t = workgroup_plan(M, N, K, sub, w8).us;
    if (us < 0 || t < us + (act_order ? 4.0 : 0.0)) { us = t; best = D2_WORKGROUP; }
  }
  if (r.us >= 0 && (us < 0 || r.us < us) && (!act_order || best == D2_WORKGROUP)) best = D2_ROWS;
  return best;
}

int decode2_launch_msp(const Decode2Params& p, int gs, int rc, bool bf16, bool zp, hipStream_t s);      // w4a16_decode2_msp.hip
int decode2_launch_msp_sub(const Decode2Params& p, int sub, int gs, bool bf16, bool zp, hipStream_t s);     // w4a16_decode2_msp_sub.hip
int decode2_launch_msp_w8(const Decode2Params& p, int sub, int gs, bool bf16, hipStream_t s);               // w4a16_decode2_msp_w8.hip

}  // namespace vaq

extern "C" int vaq_w4a16_decode_plan(int64_t size_m, int64_t size_n, int64_t size_k, int sub, int w8, int kind, double* plan) {
  using namespace vaq;
  VAQ_CHECK_ARG(size_m > 0 && size_m <= DECODE2_MAX_M_ROWS && size_n > 0 && size_n % 64 == 0 && size_k > 0 && size_k % 128 == 0 &&
                    size_n < (1 << 24) && size_k < (1 << 24) && (sub == 1 || sub == 2 || sub == 4) && plan != nullptr &&
                    (kind == 2 || size_m <= DECODE2_MAX_M), "w4a16_decode_plan: bad arguments");
  const int M = (int)size_m, N = (int)size_n, K = (int)size_k;
  Decode2Plan p;
  if (kind == 2) p = rows_plan(M, N, K, sub, w8 != 0);
  else if (kind == 0) p = workgroup_plan(M, N, K, sub, w8 != 0);
  else {
    p.c = pick_by_rule(M, N, K, sub, w8 != 0);
    p.us = decode2_us(workgroup_cost(M, sub, w8 != 0), p.c, M, N, K, sub, w8 != 0, (M + 15) / 16, 1);
  }
  const double out[6] = {(double)p.c.gs, (double)p.c.wks, (double)p.c.wn, (double)p.c.sk, (double)p.c.mr, p.us};
  for (int i = 0; i < 6; ++i) plan[i] = out[i];
  return VAQ_OK;
}

namespace vaq {

double w4a16_decode2_us(int M, int N, int K, int sub, bool w8, bool rows) {
  return (rows ? rows_plan(M, N, K, sub, w8) : workgroup_plan(M, N, K, sub, w8)).us;
}

// The same of a call of up to 32 rows with act_order, and what of it is the gather: two dependent loads and, for every 1000 elements that a compute unit's
// workgroups gather, 0.16 us (1077 timings, 18 % rms, 6 % low).
double w4a16_decode2_gather_us(int M, int N, int K, int sub, bool w8, double* gather) {
  const Decode2Plan p = workgroup_plan(M, N, K, sub, w8);
  const double wgs = (double)((N / 16 + p.c.wn - 1) / p.c.wn) * p.c.sk / num_cus_current_device();
  *gather = 0.6 + 0.159e-3 * M * 128 * p.c.gs * p.c.wks * fmax(1.0, wgs);
  return p.us + *gather;
}

int w4a16_decode2_workspace(int M, int N, int K, int sub, bool w8, size_t* c_tmp_bytes, size_t* counter_ints) {
  const Decode2Config c = workgroup_plan(M, N, K, sub, w8).c;
  const int MB = (M + 15) / 16;
  const int NT = N / 16;
  *c_tmp_bytes = c.sk > 1 ? (size_t)c.sk * NT * MB * 64 * sizeof(v4f) : 0;
  *counter_ints = c.sk > 1 ? (size_t)NT * MB : 0;
  return VAQ_OK;
}

int w4a16_decode2_launch(const void* a, int64_t lda, const int32_t* b, const void* scales, const int32_t* zeros,
                         const int32_t* perm, const void* bias, void* c, float* c_tmp, int64_t c_tmp_bytes,
                         int32_t* counters, int64_t counter_ints, int M, int N, int K, int sub, bool channelwise,
                         int wt, int dtype, bool rows, hipStream_t s) {
  const bool w8 = wt != 0;      // 8-bit weights of either kind (1: nibble planes, 2: FP8 bytes): two blocks per 128 rows
  Decode2Params p;
  p.a = (const uint16_t*)a;
  p.lda = lda;
  p.b = (const v4u*)b;
  p.scales = (const uint16_t*)scales;
  p.zeros = (const uint32_t*)zeros;
  p.perm = perm;
  p.bias = (const uint16_t*)bias;
  p.c = (uint16_t*)c;
  p.c_tmp = c_tmp;
  p.counters = counters;
  p.M = M; p.N = N; p.K = K;
  p.G = K / 128 * (w8 ? 2 : 1);
  p.NT = N / 16;
  p.GR = channelwise ? 1 : K / 128 * sub;
  p.s_stride = channelwise ? 0 : N;
  p.z_stride = channelwise ? 0 : N / 8;
  p.k_mask = 0x000f000fu;
  p.k_ex = dtype == VAQ_BF16 ? 0x43004300u : 0x64006400u;
  VAQ_CHECK_ARG(rows || M <= DECODE2_MAX_M, "w4a16_gemm(decode): %d rows without the split of the rows over workgroups", M);
  const Decode2Plan plan = rows ? rows_plan(M, N, K, sub, w8) : workgroup_plan(M, N, K, sub, w8);
  VAQ_CHECK_SUPPORTED(plan.us >= 0, "w4a16_gemm(decode): K = %d does not fit one workgroup of 16 rows", K);
  const Decode2Config cfg = plan.c;
  p.SK = cfg.sk;
  p.WKS = cfg.wks;
  p.WN = cfg.wn;
  // private activation fill (see the kernel): measured ahead only on short streams with few staged rows (4096 x 4096 at
  // M = 1 / 4: 4.53 / 4.83 -> 4.38 / 4.52 us; 14336 x 4096 at M = 4: 9.1 -> 9.3 us; with 16 staged rows, where every
  // wavefront would fetch 16 rows of its own slice: 4096 x 4096 at M = 16 5.39 -> 5.47 us, 14336 x 4096 11.08 -> 11.07 us)
  p.PRIV = (cfg.wn == 1 && perm == nullptr && cfg.mr <= 4 && cfg.gs <= 8 && tuning().exp[0] != 1) ? 1 : 0;
  const int MB = (M + 15) / 16;
  if (cfg.sk > 1) {
    VAQ_CHECK_ARG(c_tmp != nullptr && counters != nullptr, "w4a16_gemm: split-K needs c_tmp and counters");
    VAQ_CHECK_ARG(((uintptr_t)c_tmp % 16) == 0, "w4a16_gemm: c_tmp must be 16-byte aligned");
    VAQ_CHECK_ARG((uint64_t)cfg.sk * (uint64_t)p.NT * MB * 1024u < (1ull << 31), "w4a16_gemm: split-K scratch too large");
    VAQ_CHECK_ARG(counter_ints >= (int64_t)p.NT * MB,
                  "w4a16_gemm: workspace.numel = %lld is below min_workspace_size = %lld", (long long)counter_ints,
                  (long long)p.NT * MB);
    VAQ_CHECK_ARG(c_tmp_bytes >= (int64_t)cfg.sk * p.NT * MB * 1024, "w4a16_gemm: c_tmp holds %lld bytes, the K split needs %lld",
                  (long long)c_tmp_bytes, (long long)cfg.sk * p.NT * MB * 1024);
  }
  const bool bf16 = dtype == VAQ_BF16, zp = zeros != nullptr;
  int rc;
  if (rows && w8) rc = decode2_launch_msp_w8(p, sub, cfg.gs, bf16, s);
  else if (rows && sub > 1) rc = decode2_launch_msp_sub(p, sub, cfg.gs, bf16, zp, s);
  else if (rows) rc = decode2_launch_msp(p, cfg.gs, cfg.rc, bf16, zp, s);
  else if (wt == 2) rc = decode2_launch_f8(p, cfg.gs, MB, cfg.mr, bf16, s);
  else if (w8 && sub > 1) rc = decode2_launch_w8sub(p, sub, cfg.gs, MB, cfg.mr, bf16, s);
  else if (w8) rc = decode2_launch_w8(p, cfg.gs, MB, cfg.mr, bf16, s);
  else if (sub == 2) rc = decode2_launch_sub2(p, cfg.gs, MB, cfg.mr, bf16, zp, s);
  else if (sub == 4) rc = decode2_launch_sub4(p, cfg.gs, MB, cfg.mr, bf16, zp, s);
  else if (MB > 2) rc = decode2_launch_mb34(p, cfg.gs, MB, bf16, zp, s);
  else if (MB == 1) rc = dispatch_mr2<1>(p, cfg, bf16, zp, s);
  else rc = dispatch_types2<2, 16>(p, cfg.gs, cfg.rc, bf16, zp, s);
  if (rc != VAQ_OK) return rc;
  VAQ_CHECK_LAUNCH("w4a16_gemm(decode)");
  return VAQ_OK;
}

}  // namespace vaq
