// Host side of the prefill kernels (w4a16_prefill_kernel.h): tile and K-split choice, workspace sizes, launch of the
// instances for quantisation groups of 128 rows and channelwise scales.
#include "tile_plan.h"
#include "w4a16_kernels.h"
#include "w4a16_prefill_kernel.h"

namespace vaq {

// ----------------------------------------------------------------------------- host side

// tile ids: 0..2 = register-staged kernel (256x256, 128x128, 64x128); 10.. = direct-to-LDS kernel (BM x BN);
// 30 = 256 x 256 with the weights dequantised in registers (w4a16_prefill3_kernel.h)
int prefill_launch_reg(const PrefillParams& p, bool bf16, bool zp, hipStream_t s);      // w4a16_prefill3.hip

template <bool BF16, bool HAS_ZP>
static int dispatch_tile(const PrefillParams& p, int tile, hipStream_t s) {
  switch (tile) {
    case 10: return launch_prefill2<BF16, 256, 256, 2, 4, HAS_ZP, 1>(p, s);   // 8 wavefronts, 128 x 64 each
    case 20: return launch_prefill2<BF16, 256, 256, 2, 4, HAS_ZP, 1, false, true>(p, s);   // the same, alternating phases
    case 30: return prefill_launch_reg(p, BF16, HAS_ZP, s);                                // 4 wavefronts, 256 x 64 each
    case 11: return launch_prefill2<BF16, 256, 256, 2, 2, HAS_ZP, 1>(p, s);   // 4 wavefronts, 128 x 128 each
    case 12: return launch_prefill2<BF16, 128, 128, 2, 4, HAS_ZP, 1>(p, s);   // 8 wavefronts, 64 x 32 each
    case 13: return launch_prefill2<BF16, 128, 256, 2, 4, HAS_ZP, 1>(p, s);   // 8 wavefronts, 64 x 64 each
    case 14: return launch_prefill2<BF16, 64, 128, 2, 4, HAS_ZP, 1>(p, s);    // 8 wavefronts, 32 x 32 each
    case 15: return launch_prefill2<BF16, 128, 64, 2, 2, HAS_ZP, 1>(p, s);    // 4 wavefronts, 64 x 32 each
    case 16: return launch_prefill2<BF16, 256, 128, 4, 2, HAS_ZP, 1>(p, s);   // 8 wavefronts, 64 x 64 each
    case 0: return launch_prefill<BF16, 4, 4, HAS_ZP, 1>(p, s);   // 256 x 256
    case 1: return launch_prefill<BF16, 2, 2, HAS_ZP, 1>(p, s);   // 128 x 128
    case 2: return launch_prefill<BF16, 1, 2, HAS_ZP, 1>(p, s);   //  64 x 128
    default: break;
  }
  set_error("w4a16_gemm(prefill): unknown tile id %d", tile);
  return VAQ_ERR_UNSUPPORTED;
}

// Fitted to 815 problems with M = 65 .. 6000, K = 1024 .. 14336, N = 1024 .. 28672 drawn over the logarithm (4-bit codes with zero
// points, bf16), every shape and K split of each timed on cold weights.  Over the same 815 problems the plans that rules by size
// had chosen were in the mean 10 % slower than the fastest one (5 % of it the eight-wavefront shapes 12, 14 and 16 that came with
// the prices: 4096 x 4096 at M = 1024 50.7 -> 45.6 us, at M = 2048 77 -> 71 us, 4096 x 6144 at M = 333 34.6 -> 32.8 us, 4096 x 28672
// at M = 100 48.7 -> 43.1 us; nothing where the rules had the 256 x 256 tiles right, M = 4096).  Checked over 3276 problems with M = 17 ..
// 8192, K = 256 .. 28672, N = 256 .. 152064 (47137 launches, profiles/plan_prices): the cheapest plan is in the mean 1.1 % slower than
// the fastest (N > 28672 0.8 %, K or N below 1024 0.8 %, 17 .. 128 rows 1.4 - 2.0 %), 99 of 100 less than 15 %.
constexpr TileShape W4_TILE_SHAPES[] = {
    {12, 128, 128, 8, 2, 0.39, 0.578, 0.092, 0.352, 0.226}, {14, 64, 128, 8, 2, 0, 0.426, 0.041, 0.230, 0.330},
    {15, 128, 64, 4, 2, 0, 0.456, 0.025, 0.176, 0.392},     {16, 256, 128, 8, 1, 2.57, 0.764, 0.194, 0, 0.122},
    {13, 128, 256, 8, 1, 2.93, 0.869, 0.186, 0, 0.061},     {20, 256, 256, 8, 1, 6.10, 1.200, 0.422, 0, 0.024}};
constexpr TileCosts W4_TILE_COSTS = {0.277, 1.42, 0.796, 0.162, 0.0};

// Without direct-to-LDS loads (an A of 4 GiB and more): the largest register-staged tile that fills the device.
static int pick_register_staged(int M, int N) {
  const int64_t cus = num_cus_current_device();
  auto tiles = [&](int bm, int bn) { return (int64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  return tiles(256, 256) >= cus ? 0 : (tiles(128, 128) >= cus ? 1 : 2);
}

// Tile shape and K split for a problem.  `reg_ok`: 4-bit codes in groups of 128 rows or channelwise -- what the shapes 13 and 30
// are built for.
static TilePlan make_plan_prefill(int M, int N, int K, bool reg_ok) {
  const int64_t cus = num_cus_current_device();
  const int G = K / 128;
  const VaqTuning& tn = tuning();
  const int forced = tn.prefill_tile - 1;
  TilePlan best;
  // partial tiles are addressed with 32-bit offsets; the entry point on library-owned scratch says what room it has for them
  const int64_t most = tn.exp[14] > 0 ? (int64_t)tn.exp[14] * 1024 : (1ll << 32);
  for (const TileShape& t : W4_TILE_SHAPES) {
    const bool is256 = t.id == 20;
    if (forced >= 0 ? forced != t.id && !(is256 && (forced == 10 || forced == 11 || forced == 30)) : t.id == 13 && !reg_ok) continue;
    const int64_t tiles = (int64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    const int64_t rest = tiles % cus;
    auto consider = [&](int sk, int64_t tail_first) {
      consider_tile_plan(best, t, W4_TILE_COSTS, M, N, 0.5 * N * K, tiles, sk, tail_first, 2.0 * G, cus, sk > 1 ? most : 1);
    };
    if (tn.prefill_split > 0) {
      const int sk = tn.prefill_split <= G ? tn.prefill_split : G;
      consider_tile_plan(best, t, W4_TILE_COSTS, M, N, 0.5 * N * K, tiles, sk, 0, 2.0 * G, cus, 1ll << 32);
      continue;
    }
    // K in up to 8 parts of at least 3 groups, on up to 2.4 rounds of workgroups.  (All of 1 .. 8: without 5 and 7 12 % of the
    // problems had another plan, in the mean 3.2 % slower; 48 tiles fill one round in five parts only, 24576 x 6144 at M = 512
    // 154 -> 146 us, 11648 x 1984 at M = 277 27.6 -> 21.4 us)
    for (int sk = 1; sk <= 8; ++sk)
      if (sk == 1 || (G / sk >= 3 && tiles * sk * 10 <= cus * 24)) consider(sk, 0);
    // 256 x 256 tiles that end in a round of workgroups at most half full: the tiles of that round in parts of at least 8 groups
    // that fill it, the others whole (4096 x 6144 at M = 4096: 384 tiles = 256 whole + 128 in two parts each, 205 -> 189 us)
    if (is256 && tiles > cus && rest > 0 && tn.exp[6] > 1) best = TilePlan();      // (development switch: this plan alone)
    if (is256 && tiles > cus && rest > 0 && tn.exp[10] != 1)
      for (int sk : {2, 3, 4})
        if (rest * sk <= cus && (tn.exp[6] > 1 ? sk == tn.exp[6] && G / sk >= 3 : G / sk >= 8)) consider(sk, tiles - rest);
  }
  if (forced >= 0 && best.id >= 0) {
    best.id = forced;
    if (forced == 11 || forced == 30) best.nw = 4;
  } else if (best.id == 20 && best.sk == 1 && reg_ok && K >= 4096 && best.tiles * 5 >= cus * 4) {
    // Whole 256 x 256 tiles on most of the device and a long K: dequantised in registers (four wavefronts of 256 x 64), 2 % ahead
    // of the eight wavefronts with alternating phases; on a short K, with fewer tiles or with a split K 1-7 % behind.
    best.id = 30;
    best.nw = 4;
  }
  return best;
}

static TilePlan plan_prefill(int M, int N, int K, bool direct_ok, bool reg_ok) {
  const int forced = tuning().prefill_tile - 1;
  if (!direct_ok || (forced >= 0 && forced < 10)) {
    TilePlan pl;
    pl.id = forced >= 0 ? forced : pick_register_staged(M, N);
    return pl;
  }
  static thread_local TilePlanTable table;
  if (tuning_active()) return make_plan_prefill(M, N, K, reg_ok);
  return table.get(M, N, K, num_cus_current_device() * 2 + (reg_ok ? 1 : 0), [&] { return make_plan_prefill(M, N, K, reg_ok); });
}

// Predicted time of the tile kernel (negative: not known, register-staged tiles).
double w4a16_prefill_us(int M, int N, int K, bool reg_ok) { return plan_prefill(M, N, K, true, reg_ok).us; }

int w4a16_prefill_workspace(int M, int N, int K, size_t* c_tmp_bytes, size_t* counter_ints) {
  // enough for either choice of shapes: the weight format is not known here
  const TilePlan a = plan_prefill(M, N, K, true, false), b = plan_prefill(M, N, K, true, true);
  *c_tmp_bytes = (size_t)(a.tmp_bytes() > b.tmp_bytes() ? a.tmp_bytes() : b.tmp_bytes());
  *counter_ints = (size_t)(a.counter_ints() > b.counter_ints() ? a.counter_ints() : b.counter_ints());
  return VAQ_OK;
}

int w4a16_prefill_launch(const void* a, int64_t lda, const int32_t* b, const void* scales, const int32_t* zeros,
                         const void* bias, void* c, float* c_tmp, int64_t c_tmp_bytes, int32_t* counters,
                         int64_t counter_ints, int M, int N, int K, int sub, bool channelwise, int wt, int dtype,
                         hipStream_t s) {
  const bool w8 = wt != 0;      // 8-bit weights of either kind: two 1 KiB blocks per tile
  PrefillParams p;
  p.a = (const uint16_t*)a;
  p.lda = lda;
  p.b = (const v4u*)b;
  p.scales = (const uint16_t*)scales;
  p.zeros = (const uint32_t*)zeros;
  p.bias = (const uint16_t*)bias;
  p.c = (uint16_t*)c;
  p.c_tmp = c_tmp;
  p.counters = counters;
  p.M = M; p.N = N; p.K = K;
  p.G = K / 128;
  p.NT = N / 16;
  p.s_stride = channelwise ? 0 : N;
  p.z_stride = channelwise ? 0 : N / 8;
  const bool direct_ok = (uint64_t)M * (uint64_t)lda * 2 < (1ull << 32);
  if (w8 && !direct_ok) {
    set_error("w4a16_gemm(prefill): 8-bit weights with an A of 4 GiB or more are not built");
    return VAQ_ERR_UNSUPPORTED;
  }
  TilePlan pl = plan_prefill(M, N, K, direct_ok, !w8 && sub == 1);
  // A caller that passes no scratch at all gets the unsplit kernel (same result, no K split); scratch that is there but
  // too small is the caller's mistake and is reported, not worked around.
  if (pl.sk > 1 && c_tmp == nullptr && counters == nullptr) pl.sk = 1;
  // Splitting only the tiles of a half-empty last round is an optimisation that whole tiles replace at no other cost than
  // time: scratch that does not hold it (the library-owned scratch of the no-allocation entry point, say) switches it off.
  if (pl.sk > 1 && pl.tail_first > 0 && (c_tmp_bytes < pl.tmp_bytes() || counter_ints < pl.counter_ints())) pl.sk = 1;
  if (pl.sk == 1) pl.tail_first = 0;
  if (pl.sk > 1) {
    const int64_t need_tmp = pl.tmp_bytes(), need_cnt = pl.counter_ints();
    VAQ_CHECK_ARG(c_tmp != nullptr && counters != nullptr, "w4a16_gemm: split-K needs both c_tmp and counters");
    VAQ_CHECK_ARG(counter_ints >= need_cnt, "w4a16_gemm: workspace.numel = %lld is below min_workspace_size = %lld",
                  (long long)counter_ints, (long long)need_cnt);
    VAQ_CHECK_ARG(c_tmp_bytes >= need_tmp, "w4a16_gemm: c_tmp holds %lld bytes, the K split needs %lld",
                  (long long)c_tmp_bytes, (long long)need_tmp);
  }
  p.SK = pl.sk;
  p.tail_first = (int)pl.tail_first;
  const bool bf16 = dtype == VAQ_BF16, zp = zeros != nullptr;
  int rc;
  // the alternating-phase and the register-dequantising variants exist for 4-bit codes in groups of 128 rows / channelwise
  const int tile_other = (pl.id == 20 || pl.id == 30) ? 10 : pl.id;
  if (wt == 2) rc = prefill_launch_f8(p, tile_other, bf16, s);
  else if (w8) rc = prefill_launch_w8(p, sub, tile_other, bf16, s);
  else if (sub > 1) rc = prefill_launch_sub(p, sub, tile_other, bf16, zp, s);
  else if (bf16) rc = zp ? dispatch_tile<true, true>(p, pl.id, s) : dispatch_tile<true, false>(p, pl.id, s);
  else rc = zp ? dispatch_tile<false, true>(p, pl.id, s) : dispatch_tile<false, false>(p, pl.id, s);
  if (rc != VAQ_OK) return rc;
  VAQ_CHECK_LAUNCH("w4a16_gemm(prefill)");
  return VAQ_OK;
}

}  // namespace vaq
