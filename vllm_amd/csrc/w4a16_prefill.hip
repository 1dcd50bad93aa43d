// Host side of the prefill kernels (w4a16_prefill_kernel.h): tile and K-split choice, workspace sizes, launch of the
// instances for quantisation groups of 128 rows and channelwise scales.
#include "tile_plan.h"
#include "w4a16_kernels.h"
#include "w4a16_prefill_kernel.h"

#include <iterator>

namespace vaq {

// ----------------------------------------------------------------------------- host side

// tile ids: 0..2 = register-staged kernel (256x256, 128x128, 64x128); 10.. = direct-to-LDS kernel (BM x BN);
// 41.. = strips (w4a16_strip_kernel.h), 48 = w4a16_tile256_kernel.h
// w4a16_strip*.hip
int prefill_launch_strip(const PrefillParams& p, int tile, bool bf16, bool zp, hipStream_t s);
int prefill_launch_strip_sub(const PrefillParams& p, int sub, int tile, bool bf16, bool zp, hipStream_t s);
int prefill_launch_strip_w8(const PrefillParams& p, int sub, int tile, bool bf16, hipStream_t s);
// w4a16_tile256*.hip (id 48)
int prefill_launch_tile256(const PrefillParams& p, bool bf16, bool zp, hipStream_t s);
int prefill_launch_tile256_sub(const PrefillParams& p, int sub, bool bf16, bool zp, hipStream_t s);
int prefill_launch_tile256_w8(const PrefillParams& p, int sub, bool bf16, hipStream_t s);

template <bool BF16, bool HAS_ZP>
static int dispatch_tile(const PrefillParams& p, int tile, hipStream_t s) {
  switch (tile) {
    case 10: return launch_prefill2<BF16, 256, 256, 2, 4, HAS_ZP, 1>(p, s);   // 8 wavefronts, 128 x 64 each
    case 20: return launch_prefill2<BF16, 256, 256, 2, 4, HAS_ZP, 1, false, true>(p, s);   // the same, alternating phases
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

// What the tile shapes cost, by weight format (tile_plan.h).
// 4-bit codes: fitted to 2712 problems with M = 17 .. 8192, half of them with K = 1024 .. 14336 and N = 1024 .. 28672, half with K =
// 256 .. 28672 and N = 256 .. 152064, drawn over the logarithm, every shape and K split of each timed on cold weights (104302
// launches, profiles/plan_prices; bf16, zero points).  The cheapest plan is in the mean 0.7 % slower than the fastest, 99 of 100 less
// than 10 %, as over a half of the layers that a fit to the other half had not seen.  The fastest plan of the shapes
// 12 .. 20 (weights through LDS) takes this much more than that of the shapes from 41 on (strips): 41 / 29 / 26 / 22 / 17 / 11 / 8 / 3 %
// at M up to 32 / 64 / 128 / 256 / 512 / 1024 / 2048 / 8192; at M > 512 it is ahead in 10-25 % of the problems, by a few percent.
// The shape 48 (w4a16_tile256_kernel.h; before it a 256 x 256 shape of the strip kernel, for 4-bit codes in groups of 128 rows alone) came later, in all four tables, timed on
// their problems of more than 128 rows; its constants, and with them those of 8-bit codes and of five other large shapes in groups of 64 / 32 rows of 4 bits, are those whose choice loses
// least.  Over 4581 other problems of M = 200 .. 8192 it is the fastest plan of 47 %, and what it takes there is 0.92 (4 bits in groups of 128 rows) .. 0.88 of what those problems took.
constexpr TileShape W4_TILE_SHAPES[] = {
    {12, 128, 128, 8, 2, 0.536, 0.606, 0.0793, 0.375, 0.153}, {14, 64, 128, 8, 2, 0, 0.535, 0.0271, 0.177, 0.252},
    {15, 128, 64, 4, 2, 0, 0.553, 0.0166, 0.0944, 0.337},     {16, 256, 128, 8, 1, 1.88, 0.781, 0.176, 0, 0.0912},
    {13, 128, 256, 8, 1, 2.36, 0.829, 0.193, 0, 0.0731},      {20, 256, 256, 8, 1, 3.75, 1.23, 0.279, 0, 0.0186},
    {41, 32, 128, 8, 2, 1.99, 0.202, 0.0375, 0.163, 0.118},   {51, 32, 64, 8, 2, 1.43, 0.104, 0.0134, 0.148, 0.399},
    {42, 64, 128, 8, 2, 2.44, 0.233, 0.0366, 0.25, 0.116},    {52, 64, 64, 8, 1, 2.68, 0.138, 0.0327, 0, 0.0886},
    {43, 96, 128, 8, 1, 3.1, 0.266, 0.085, 0, 0.169},         {44, 128, 128, 8, 1, 3.63, 0.328, 0.114, 0, 0.126},
    {46, 128, 256, 8, 1, 3.64, 0.495, 0.324, 0, 0.0655},      {66, 128, 256, 8, 1, 6.38, 0.566, 0.164, 0, 0.119},
    {48, 256, 256, 4, 1, 5.52, 1.09, 0.156, 0, 0.0428}};
constexpr TileCosts W4_TILE_COSTS = {0.163, 0.628, 0.63, 0.253, 0.0};
// Groups of 64 / 32 rows: 2744 such problems, 78807 launches (64 rows with zero points, 32 without and with, these in fp16 too).  One workgroup of
// the shape 42 to a compute unit: its scales of the sub-groups leave no room for a second one in the registers.  In the mean 0.6 % on layers
// that a fit to the other half had not seen (0.45, 0.3, 0.55 and 1.05 % over the four; with the constants above and their two workgroups
// 0.7, 0.7, 1.0 and 1.9 %).
constexpr TileShape W4SUB_TILE_SHAPES[] = {
    {12, 128, 128, 8, 2, 0.726, 0.631, 0.0892, 0.392, 0.139}, {14, 64, 128, 8, 2, 0, 0.613, 0.0195, 0.177, 0.269},
    {15, 128, 64, 4, 2, 0, 0.583, 0.0117, 0.107, 0.358},      {16, 256, 128, 8, 1, 1.66, 0.83, 0.166, 0, 0.0983},
    {20, 256, 256, 8, 1, 4.63, 1.36, 0.123, 0, 0.0118},
    {41, 32, 128, 8, 2, 2.38, 0.236, 0.0194, 0.195, 0.161},   {51, 32, 64, 8, 2, 1.31, 0.124, 0.00437, 0.141, 0.681},
    {42, 64, 128, 8, 1, 2.47, 0.264, 0.0529, 0, 0.0702},      {52, 64, 64, 8, 1, 2.52, 0.165, 0.0145, 0, 0.067},
    {43, 96, 128, 8, 1, 2.31, 0.334, 0.0356, 0, 0.27},       {44, 128, 128, 8, 1, 3.2, 0.381, 0.0552, 0, 0.242},
    {46, 128, 256, 8, 1, 3.88, 0.573, 0.233, 0, 0.0539},
    {48, 256, 256, 4, 1, 7.4, 1.2, 0.0749, 0, 0.0156}};
constexpr TileCosts W4SUB_TILE_COSTS = {0.131, 0.547, 0.631, 0.274, 0.0};
// What the kernel with activations in registers is weighed against (w4a16_tile_us): the strips ahead of that shape, at the prices that its shares (w4a16_gemm.hip) were set at.  Five large shapes
// followed the shape 48, for 0.02 .. 0.06 % of what the choice among tiles loses; at those 14 of 29310 drawn problems of 17 .. 256 rows would leave that kernel, which rounds less.
constexpr TileShape W4SUB_WEIGHED_SHAPES[] = {
    {12, 128, 128, 8, 2, 0.726, 0.631, 0.0892, 0.392, 0.139}, {14, 64, 128, 8, 2, 0, 0.613, 0.0195, 0.177, 0.269},
    {15, 128, 64, 4, 2, 0, 0.583, 0.0117, 0.107, 0.358},      {16, 256, 128, 8, 1, 1.95, 0.825, 0.183, 0, 0.11},
    {20, 256, 256, 8, 1, 4.48, 1.36, 0.12, 0, 0.013},
    {41, 32, 128, 8, 2, 2.38, 0.236, 0.0194, 0.195, 0.161},   {51, 32, 64, 8, 2, 1.31, 0.124, 0.00437, 0.141, 0.681},
    {42, 64, 128, 8, 1, 2.47, 0.264, 0.0529, 0, 0.0702},      {52, 64, 64, 8, 1, 2.52, 0.165, 0.0145, 0, 0.067},
    {43, 96, 128, 8, 1, 2.57, 0.333, 0.0362, 0, 0.257},       {44, 128, 128, 8, 1, 3.05, 0.386, 0.0558, 0, 0.246},
    {46, 128, 256, 8, 1, 3.85, 0.584, 0.219, 0, 0.0488}};
// 8-bit codes, whose dequantisation takes longer: 1216 such problems, 37199 launches, in the mean 0.6 % (2.4 % with the first constants above).
// Groups of 64 rows take them too, but for the slots of the shape 41 (make_plan_prefill): 876 problems, 24724 launches, 0.35 %.
// The strips that read activation fragments two slices ahead (w4a16_strip_kernel.h: the shapes 42 in groups of 64 rows and more, 43, 44, 46) take 0.94 .. 0.98 of what these problems were
// timed at first.  All constants of 8-bit codes follow: with those before, 0.9 / 0.65 / 1.07 % in groups of 128 / 64 / 32 rows; 420 drawn calls of M = 33 .. 6500 take 0.997 in the
// mean of their time with those (25 of them more than 3 % faster, 9 slower).
constexpr TileShape W8_TILE_SHAPES[] = {
    {12, 128, 128, 8, 2, 0.789, 0.614, 0.0538, 0.433, 0.0931}, {14, 64, 128, 8, 2, 0.012, 0.602, 0.0299, 0.164, 0.233},
    {15, 128, 64, 4, 2, 0.00863, 0.61, 0.0136, 0.0904, 0.301},  {16, 256, 128, 8, 1, 1.57, 0.886, 0.136, 0, 0.0688},
    {20, 256, 256, 8, 1, 4.2, 1.23, 0.29, 0, 0.0258},
    {41, 32, 128, 8, 2, 4.05, 0.252, 0.0252, 0.241, 0.12},    {51, 32, 64, 8, 1, 2.05, 0.174, 0.013, 0, 0.664},
    {42, 64, 128, 8, 1, 2.85, 0.306, 0.046, 0, 0.103},        {52, 64, 64, 8, 1, 2.54, 0.194, 0.0205, 0, 0.0657},
    {43, 96, 128, 8, 1, 3.43, 0.339, 0.0444, 0, 0.39},        {44, 128, 128, 8, 1, 4.19, 0.403, 0.062, 0, 0.157},
    {46, 128, 256, 8, 1, 4.46, 0.629, 0.162, 0, 0.102},
    {48, 256, 256, 4, 1, 8.97, 1.07, 0.162, 0, 0.0335}};
constexpr TileCosts W8_TILE_COSTS = {0.176, 0.376, 0.706, 0.291, 0.0};
// Groups of 32 rows: 1549 such problems, 45867 launches, in bf16 and fp16, whose strips convert code by code here; in the mean 0.67 % (with the constants above
// 1 in 8 fp16 problems more than 5 % behind).
constexpr TileShape W8G32_TILE_SHAPES[] = {
    {12, 128, 128, 8, 2, 0.475, 0.714, 0.0654, 0.436, 0.104},  {14, 64, 128, 8, 2, 0.00821, 0.605, 0.0188, 0.298, 0.273},
    {15, 128, 64, 4, 2, 0.0146, 0.626, 0.0107, 0.207, 0.296},  {16, 256, 128, 8, 1, 2.08, 0.962, 0.141, 0, 0.0507},
    {20, 256, 256, 8, 1, 4.52, 1.38, 0.228, 0, 0.0128},
    {41, 32, 128, 8, 1, 2.87, 0.391, 0.0367, 0, 0.0948},        {51, 32, 64, 8, 1, 1.07, 0.196, 0.00868, 0, 0.29},
    {42, 64, 128, 8, 1, 2.89, 0.381, 0.0473, 0, 0.0972},       {52, 64, 64, 8, 1, 2.41, 0.214, 0.0107, 0, 0.105},
    {43, 96, 128, 8, 1, 1.95, 0.429, 0.0229, 0, 0.373},        {44, 128, 128, 8, 1, 4.55, 0.455, 0.039, 0, 0.449},
    {46, 128, 256, 8, 1, 3.74, 0.796, 0.109, 0, 0.164},
    {48, 256, 256, 4, 1, 7.26, 1.34, 0.129, 0, 0.00143}};
constexpr TileCosts W8G32_TILE_COSTS = {0.146, 0.456, 0.643, 0.288, 0.0};
// The shapes with weights through LDS by themselves, fitted to 815 problems of 4-bit codes: what FP8 weights are built for (but 13),
// and the price that up to 256 rows are weighed against the decode kernels at (w4a16_staged_us).
constexpr TileShape LDS_TILE_SHAPES[] = {
    {12, 128, 128, 8, 2, 0.39, 0.578, 0.092, 0.352, 0.226}, {14, 64, 128, 8, 2, 0, 0.426, 0.041, 0.230, 0.330},
    {15, 128, 64, 4, 2, 0, 0.456, 0.025, 0.176, 0.392},     {16, 256, 128, 8, 1, 2.57, 0.764, 0.194, 0, 0.122},
    {13, 128, 256, 8, 1, 2.93, 0.869, 0.186, 0, 0.061},     {20, 256, 256, 8, 1, 6.10, 1.200, 0.422, 0, 0.024}};
constexpr TileCosts LDS_TILE_COSTS = {0.277, 1.42, 0.796, 0.162, 0.0};
static_assert(W4_TILE_SHAPES[std::size(W4_TILE_SHAPES) - 1].id == 48 && std::size(W4SUB_WEIGHED_SHAPES) == std::size(W4SUB_TILE_SHAPES) - 1 &&
                  W8_TILE_SHAPES[std::size(W8_TILE_SHAPES) - 1].id == 48 && W8G32_TILE_SHAPES[std::size(W8G32_TILE_SHAPES) - 1].id == 48,
              "what the kernel with activations in registers is weighed against is known ahead of the last shape");
struct TilePrices {
  const TileShape *begin, *end;
  const TileCosts& costs;
  double weight_bytes;      // per element, as the fit counted them
};
static TilePrices tile_prices(TileFormat format) {
  if (format == TILES_SUB_WEIGHED) return {std::begin(W4SUB_WEIGHED_SHAPES), std::end(W4SUB_WEIGHED_SHAPES), W4SUB_TILE_COSTS, 0.5};
  if (format == TILES_SUB) return {std::begin(W4SUB_TILE_SHAPES), std::end(W4SUB_TILE_SHAPES), W4SUB_TILE_COSTS, 0.5};
  if (format == TILES_8BIT_32) return {std::begin(W8G32_TILE_SHAPES), std::end(W8G32_TILE_SHAPES), W8G32_TILE_COSTS, 1.0};
  if (format == TILES_8BIT || format == TILES_8BIT_64) return {std::begin(W8_TILE_SHAPES), std::end(W8_TILE_SHAPES), W8_TILE_COSTS, 1.0};
  if (format == TILES_FP8 || format == TILES_PLAIN_STAGED) return {std::begin(LDS_TILE_SHAPES), std::end(LDS_TILE_SHAPES), LDS_TILE_COSTS, 0.5};
  return {std::begin(W4_TILE_SHAPES), std::end(W4_TILE_SHAPES), W4_TILE_COSTS, 0.5};
}

// Without direct-to-LDS loads (an A of 4 GiB and more): the largest register-staged tile that fills the device.
static int pick_register_staged(int M, int N) {
  const int64_t cus = num_cus_current_device();
  auto tiles = [&](int bm, int bn) { return (int64_t)((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  return tiles(256, 256) >= cus ? 0 : (tiles(128, 128) >= cus ? 1 : 2);
}

// One or two tiles one below the other, up to 512 rows, the shape 48 takes 4 .. 10 % longer beside the others than its constants say, which are fitted to thousands of rows too.  Of the recorded
// problems of 129 .. 256 rows the chosen plan takes 1.0072 -> 1.0066 of the fastest one's time (4 bits, groups of 128), 1.0077 -> 1.0065 (8 bits) and 1.0037 -> 1.0031 (groups of 64); from 257 to
// 512 1.0071, 1.0084 -> 1.0083 and 1.0050 -> 1.0048.  90 drawn calls whose plan moves by it take 0.957 of the time, 63 more than 3 % faster, 3 slower (4 % at most); 8 bits, 9856 x 23488 at
// M = 313 227 -> 203 us, 1280 x 24384 at M = 365 in groups of 64 38.7 -> 36.2.  Not in smaller groups, whose recorded choice it makes no better (fp16 up to 15 % slower).
constexpr double TILE256_FEW_ROWS_PRICE = 1.03;

// Tile shape and K split for a problem (the shapes 13 and 66 are built for TILES_PLAIN; 30, another kernel of the shape 20 in
// recorded timings, stands for 20).
static TilePlan make_plan_prefill(int M, int N, int K, TileFormat format) {
  const int64_t cus = num_cus_current_device();
  const int G = K / 128;
  const VaqTuning& tn = tuning();
  const int forced = tn.prefill_tile == 31 ? 20 : tn.prefill_tile - 1;
  const bool plain = format == TILES_PLAIN || format == TILES_PLAIN_STAGED;
  const TilePrices prices = tile_prices(format);
  const double weight_bytes = prices.weight_bytes * N * K;
  TilePlan best;
  // partial tiles are addressed with 32-bit offsets; the entry point on library-owned scratch says what room it has for them
  const int64_t most = tn.exp[14] > 0 ? (int64_t)tn.exp[14] * 1024 : (1ll << 32);
  for (const TileShape* shape = prices.begin; shape != prices.end; ++shape) {
    TileShape t = *shape;
    if (t.id == 41 && format == TILES_8BIT_64) t.slots = 1;      // (133 registers)
    if (t.id == 48 && M <= 512 && (format == TILES_PLAIN || format == TILES_8BIT || format == TILES_8BIT_64)) {
      t.base *= TILE256_FEW_ROWS_PRICE;
      t.step *= TILE256_FEW_ROWS_PRICE;
      t.load *= TILE256_FEW_ROWS_PRICE;
    }
    const bool is256 = t.id == 20 || t.id == 48;
    if (t.id == 48) best.us_strips = best.us;      // (the last row of a table)
    if (forced >= 0 ? forced != t.id && !(t.id == 20 && (forced == 10 || forced == 11)) : (t.id == 13 || t.id == 66) && !plain) continue;
    const int64_t tiles = (int64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    const int64_t rest = tiles % cus;
    auto consider = [&](int sk, int64_t tail_first) {
      consider_tile_plan(best, t, prices.costs, M, N, weight_bytes, tiles, sk, tail_first, 2.0 * G, cus, sk > 1 ? most : 1);
    };
    if (tn.prefill_split > 0) {
      const int sk = tn.prefill_split <= G ? tn.prefill_split : G;
      consider_tile_plan(best, t, prices.costs, M, N, weight_bytes, tiles, sk, 0, 2.0 * G, cus, 1ll << 32);
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
  if (best.us_strips < 0) best.us_strips = best.us;
  if (forced >= 0 && best.id >= 0) {
    best.id = forced;
    if (forced == 11) best.nw = 4;
  }
  return best;
}

static TilePlan plan_prefill(int M, int N, int K, bool direct_ok, TileFormat format) {
  const VaqTuning& tn = tuning();
  const int forced = tn.prefill_tile - 1;
  if (!direct_ok || (forced >= 0 && forced < 10)) {
    TilePlan pl;
    pl.id = forced >= 0 ? forced : pick_register_staged(M, N);
    return pl;
  }
  // The entry point on library-owned scratch sets exp[10] and exp[14] on every call: they are part of the key, so that its calls find
  // their plans too (six to ten of them a call at 17 .. 256 rows, 0.5 - 1 us each to make).
  constexpr int KIB_MAX = 1 << 15;
  static thread_local TilePlanTable table;
  if (forced >= 0 || tn.prefill_split > 0 || tn.exp[6] > 1 || tn.exp[14] < 0 || tn.exp[14] >= KIB_MAX) return make_plan_prefill(M, N, K, format);
  const int key = ((num_cus_current_device() * 2 + (tn.exp[10] == 1 ? 1 : 0)) * KIB_MAX + tn.exp[14]) * 8 + format;
  return table.get(M, N, K, key, [&] { return make_plan_prefill(M, N, K, format); });
}

// Predicted time of the tile kernel whose weights pass through LDS (negative: not known, register-staged tiles): what the decode
// kernels are weighed against.  The strips are faster than that, but both tile kernels round the scaled weights to 16 bits and the
// decode kernels keep their scales in fp32: problems go from these to the strips only where they went to a tile kernel before there
// were strips.
double w4a16_staged_us(int M, int N, int K, bool plain) { return plan_prefill(M, N, K, true, plain ? TILES_PLAIN_STAGED : TILES_FP8).us; }

// What the kernel with activations in registers is weighed against.  That keeps its codes exact and its scales in fp32, the tile kernels round each scaled weight to 16 bits: like
// above, no call loses those bits to the 256 x 256 tiles, which came last and are cheaper than the strips from 130 rows on where K N is large (6 of 6677 problems of
// 17 .. 256 rows of 4-bit codes in groups of 128, 28 and 2 in groups of 64 and 32 had gone, at the prices of two steps; 21760 x 12096 at M = 157 is priced 105.8 there, 111.5 in such
// tiles and 117.7 in strips).
double w4a16_tile_us(int M, int N, int K, TileFormat format) { return plan_prefill(M, N, K, true, format == TILES_SUB ? TILES_SUB_WEIGHED : format).us_strips; }

int w4a16_prefill_workspace(int M, int N, int K, TileFormat format, size_t* c_tmp_bytes, size_t* counter_ints) {
  const TilePlan pl = plan_prefill(M, N, K, true, format);
  *c_tmp_bytes = (size_t)pl.tmp_bytes();
  *counter_ints = (size_t)pl.counter_ints();
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
  TilePlan pl = plan_prefill(M, N, K, direct_ok, tile_format(sub, wt));
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
  // the alternating-phase variant exists for 4-bit codes in groups of 128 rows / channelwise
  const int tile_other = pl.id == 20 ? 10 : pl.id;
  if (pl.id == 48) {
    if (w8) rc = prefill_launch_tile256_w8(p, sub, bf16, s);
    else if (sub > 1) rc = prefill_launch_tile256_sub(p, sub, bf16, zp, s);
    else rc = prefill_launch_tile256(p, bf16, zp, s);
  } else if (pl.id > 40) {
    if (w8) rc = prefill_launch_strip_w8(p, sub, pl.id, bf16, s);
    else if (sub > 1) rc = prefill_launch_strip_sub(p, sub, pl.id, bf16, zp, s);
    else rc = prefill_launch_strip(p, pl.id, bf16, zp, s);
  } else if (wt == 2) rc = prefill_launch_f8(p, tile_other, bf16, s);
  else if (w8) rc = prefill_launch_w8(p, sub, tile_other, bf16, s);
  else if (sub > 1) rc = prefill_launch_sub(p, sub, tile_other, bf16, zp, s);
  else if (bf16) rc = zp ? dispatch_tile<true, true>(p, pl.id, s) : dispatch_tile<true, false>(p, pl.id, s);
  else rc = zp ? dispatch_tile<false, true>(p, pl.id, s) : dispatch_tile<false, false>(p, pl.id, s);
  if (rc != VAQ_OK) return rc;
  VAQ_CHECK_LAUNCH("w4a16_gemm(prefill)");
  return VAQ_OK;
}

}  // namespace vaq

extern "C" int vaq_w4a16_tile_plan(int64_t size_m, int64_t size_n, int64_t size_k, int sub, int wt, int staged, double* plan) {
  using namespace vaq;
  VAQ_CHECK_ARG(size_m > 0 && size_m < (1ll << 31) && size_n > 0 && size_n % 64 == 0 && size_n < (1 << 24) && size_k > 0 &&
                    size_k % 128 == 0 && size_k < (1 << 24) && (sub == 1 || sub == 2 || sub == 4) && wt >= 0 && wt <= 2 && plan != nullptr,
                "w4a16_tile_plan: bad arguments");
  const TileFormat format = staged ? (sub == 1 && wt == 0 ? TILES_PLAIN_STAGED : TILES_FP8) : tile_format(sub, wt);
  const TilePlan pl = plan_prefill((int)size_m, (int)size_n, (int)size_k, true, format);
  const double out[4] = {(double)pl.id, (double)pl.sk, (double)pl.tail_first, pl.us};
  for (int i = 0; i < 4; ++i) plan[i] = out[i];
  return VAQ_OK;
}
