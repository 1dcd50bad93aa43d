// Host side of the W4A16 kernel with activations in registers (w4a16_regs_kernel.h): choice of the plan, workspace sizes, launch.
#include "tile_plan.h"
#include "w4a16_kernels.h"
#include "w4a16_regs_kernel.h"

namespace vaq {

struct RegsPlan {
  int nw = 0, j = 0, mb = 0, sk = 1, rb = 1;
  double us = -1;      // predicted; negative: no plan
  size_t tmp_bytes(int N) const { return sk > 1 ? (size_t)sk * (N / 16) * rb * mb * 1024 : 0; }
  size_t counter_ints(int N) const { return sk > 1 ? (size_t)(N / 16) * rb * mb : 0; }
};

// What a launch costs, in us.  A k-tile of a wavefront: `latency`, or the arithmetic of all wavefronts that share a SIMD -- `row` per
// m-block (operands and row sums), `tile` + `tile_mb` per m-block for each n-tile; times `alone` where one wavefront has a SIMD to itself, so
// that nothing runs beside its waits, times `copies` where the sums do not fit the vector registers -- or `kb` per KB of operands that
// come into the compute unit; times `k1024` where K is a multiple of 1024 and the rows of activations and strips of weights start on the same
// memory channels.  A workgroup: `round`, its k-tiles, and the meeting of the sums, `meet` + `meet_wave` per wavefront on the compute unit for each 16 x
// 16 result.  A started round of workgroups beyond the first counts by `last` beyond its share.  Beside that the weights from memory (`mem_mb` per MB, and `again` of
// that for every further block of rows); `base` and `out` per MB of results a launch; K in parts: `handover` + per part `part` + `part_mb` per MB
// of partial results.
// Fitted, a set per format (4-bit codes in groups of 128 rows: another for up to 4 rows), to the cold times of 2.2e5 launches: 11400 problems of random layers, half of them with K 1024 .. 14336 and N
// 1024 .. 28672, half with K 256 .. 28672 and N 256 .. 152064, 1 .. 200 rows, with and without zero points, bf16 and fp16, each with up to 24
// plans (a part of those in profiles/plan_prices).  The cheapest plan takes 1.012 .. 1.015 of the fastest one's time in the mean.  8-bit codes again, after their planes became one
// operand, to 24326 launches of 1261 problems, which take 0.80 .. 0.97 of the time: cheapest plan 1.011 / 1.012 / 1.013 in groups of 128 / 64 / 32 rows (1.018 / 1.017 / 1.014 with the
// constants before), choice between this kernel and the others 1.003 / 1.002 / 1.003 of the faster one's time (1.010 / 1.008 / 1.013); 400 drawn calls of 1 .. 256 rows 0.986 by the constants,
// 5 of them more than 3 % slower, 47 faster.
struct RegsCost {
  double base, round, latency, row, tile, tile_mb, kb, mem_mb, last, meet, meet_wave, out, handover, part, part_mb, again, alone, copies, k1024;
};
constexpr RegsCost REGS_COST_W4_4ROWS = {1.81, 0.102, 0.271, 0, 0.0698, 0.0322, 0.0186, 0.137, 0.0141, 0.13, 0.0109, 2.41, 0.658, 0.334, 0.844, 0.1, 1.52, 1.2, 1.12};
constexpr RegsCost REGS_COST_W4 = {1.92, 0.0921, 0.156, 0.0473, 0.0944, 0.0133, 0.0121, 0.162, 0.069, 0.198, 0, 0.134, 0.42, 0.39, 0.893, 0.163, 1.32, 1.18, 1.08};
constexpr RegsCost REGS_COST_W4_64 = {2.13, 0.00844, 0.197, 0.0341, 0.102, 0.0279, 0.0118, 0.158, 0.121, 0.155, 0.012, 0.0826, 0.463, 0.358, 0.884, 0.173, 1.55, 1.15, 1.09};
constexpr RegsCost REGS_COST_W4_32 = {2.19, 0, 0.264, 0.00999, 0.127, 0.0499, 0.0136, 0.185, 0.0443, 0.127, 0.0131, 0.142, 0.496, 0.351, 0.912, 0.0388, 1.7, 1.01, 1.08};
constexpr RegsCost REGS_COST_W8 = {1.75, 0.00662, 0.0353, 0.00418, 0.0821, 0.021, 0.0113, 0.167, 0.00427, 0.228, 0.00326, 0.101, 0.524, 0.266, 0.925, 0.15, 1.01, 0.879, 1.07};
constexpr RegsCost REGS_COST_W8_64 = {1.94, 0.00969, 0.157, 0.00336, 0.0761, 0.0347, 0.0117, 0.161, 0.0112, 0.113, 0.00298, 0.186, 0.84, 0.348, 0.784, 0.192, 1.14, 1.05, 0.989};
constexpr RegsCost REGS_COST_W8_32 = {1.43, 0.00318, 0.38, 0.00372, 0.0848, 0.0367, 0.0136, 0.198, 0.00257, 0.166, 0.0167, 0.0899, 0.925, 0.234, 0.884, 0.128, 1.6, 0.869, 0.94};

static double regs_us(const RegsPlan& p, int M, int N, int K, int sub, bool w8, int cus) {
  const RegsCost& c = w8 ? (sub == 1 ? REGS_COST_W8 : sub == 2 ? REGS_COST_W8_64 : REGS_COST_W8_32)
                         : (sub == 1 ? (M <= 4 ? REGS_COST_W4_4ROWS : REGS_COST_W4) : sub == 2 ? REGS_COST_W4_64 : REGS_COST_W4_32);
  // (all counts fit 32 bits: at most 16 blocks of rows, 2^20 n-tiles)
  const int planes = w8 ? 2 : 1, mr = M <= 4 && p.mb == 1 ? 4 : 16;
  const int registers = regs_estimate(p.mb, p.j, sub, w8);
  const int by_lds = 160 * 1024 / (int)regs_lds_bytes(p.mb, mr, p.j, p.nw, sub, false);
  int slots = registers >= 512 ? 1 : 512 / registers > 8 ? 8 : 512 / registers;
  slots = slots * 4 / p.nw < by_lds ? slots * 4 / p.nw : by_lds;
  if (slots < 1) slots = 1;
  const int per_cu = ((N / 16 + p.j - 1) / p.j * p.rb * p.sk + cus - 1) / cus;
  const double side = per_cu < slots ? per_cu : slots, even = (double)per_cu / slots, waves = side * p.nw / 4.0;
  const double rounds = per_cu > slots ? even + c.last * ((per_cu + slots - 1) / slots - even) : 1.0;
  const int tiles = ((K / 128 + p.sk - 1) / p.sk + p.nw - 1) / p.nw;
  const double work = waves * (c.row * p.mb * (sub == 4 ? 2 : 1) + p.j * planes * (c.tile + c.tile_mb * p.mb)) * (registers > 256 ? c.copies : 1.0) *
                      (waves <= 1 ? c.alone : 1.0);
  const double bytes = c.kb * side * p.nw * (p.mb * mr * 0.25 + p.j * planes);
  const double tile = cbrt(c.latency * c.latency * c.latency + work * work * work + bytes * bytes * bytes) * (K % 1024 == 0 ? c.k1024 : 1.0);
  const double core = rounds * (c.round + tiles * tile + p.j * p.mb * (c.meet + c.meet_wave * side * p.nw));
  const double mem = c.mem_mb * 0.5e-6 * (double)K * N * planes * (1 + c.again * (p.rb - 1));
  double us = c.base + cbrt(core * core * core + mem * mem * mem) + c.out * 2e-6 * (double)M * N;
  if (p.sk > 1) us += c.handover + p.sk * (c.part + c.part_mb * 4e-6 * (double)(p.rb * 16 * p.mb) * N);
  return us;
}

// 8-bit codes, one n-tile to a wavefront, K in nine turns and more, no second workgroup on any compute unit: 4 KB of weights in flight for each wavefront do not cover the latency of that many
// turns, which takes 1.12 .. 1.18 of the price where other plans take 1.0 .. 1.05.  K is weighed in parts, or more n-tiles, as if that were 8 % more.  Of drawn calls of 1 .. 256 rows 0.8 %
// move by it; 115 of those, both plans timed, take 0.950 of the time, 74 more than 3 % less, 11 more (8 % at most).  Not in groups of 32 rows beyond 4 rows, whose arithmetic
// takes longer than that (32 such calls 1.001, 8 more than 3 % slower, 6 faster), and not from seven turns on.  9344 x 2304 at M = 15 10.05 -> 8.8 us (one n-tile, K whole -> two, three parts).
constexpr int LONG_STREAM_TURNS = 9;
constexpr double LONG_STREAM_PRICE = 1.08;

// exp[8]: 1 never this kernel, else a plan: n-tiles | m-blocks << 4 | wavefronts << 8 | parts of K << 12
static RegsPlan make_regs_plan(int M, int N, int K, int sub, bool w8) {
  const int G = K / 128, NT = N / 16, cus = num_cus_current_device();
  const int forced = tuning().exp[8];
  RegsPlan best;
  double best_us = -1;
  for (int nw : {4, 8})
    for (int mb = 1; mb <= 3; ++mb)
      for (int j = 1; j <= 8; ++j) {
        if (!regs_built(mb, j, nw, sub, w8)) continue;
        // K in up to 8 parts of a k-tile per wavefront and more where the workgroups do not fill the device, on up to two per compute unit, within
        // the library-owned scratch and the counters that a layer has (four per 16 columns, at least 4096).  (On up to 2.7, filled or not: a
        // tenth more plans, 0.02 % in the mean.)
        const int rb = (M + mb * 16 - 1) / (mb * 16), units = (NT + j - 1) / j * rb;
        for (int sk = 1; sk <= 8; ++sk) {
          RegsPlan p;
          p.nw = nw; p.j = j; p.mb = mb; p.sk = sk; p.rb = rb;
          if (forced > 1 && forced != (j | mb << 4 | nw << 8 | sk << 12)) continue;
          if (sk > 1 && forced <= 1 && (units >= cus || units * sk > 2 * cus)) break;
          if (sk > 1 && (G / sk < nw || p.tmp_bytes(N) > VAQ_STATIC_SCRATCH_DATA_BYTES || p.counter_ints(N) > (size_t)(NT > 1024 ? NT * 4 : 4096))) break;
          p.us = regs_us(p, M, N, K, sub, w8, cus);
          const double us = p.us * (w8 && (sub < 4 || M <= 4) && j == 1 && units * sk <= cus && ((G + sk - 1) / sk + nw - 1) / nw >= LONG_STREAM_TURNS ? LONG_STREAM_PRICE : 1.0);
          if (best.us < 0 || us < best_us) {
            best = p;
            best_us = us;
          }
        }
      }
  return best;
}

static RegsPlan regs_plan(int M, int N, int K, int sub, bool w8) {
  static thread_local PlanTable<RegsPlan> table;
  if (tuning().exp[8] > 1) return make_regs_plan(M, N, K, sub, w8);
  return table.get(M, N, K, (num_cus_current_device() * 8 + sub) * 2 + (w8 ? 1 : 0), [&] { return make_regs_plan(M, N, K, sub, w8); });
}

double w4a16_regs_us(int M, int N, int K, int sub, int wt, int* n_tiles, int* wavefronts) {
  // 32-bit offsets with the top bit to spare: it is what a request for nothing sets
  if (M > REGS_MAX_M || wt == 2 || (uint64_t)K * N / (wt == 1 ? 1 : 2) >= (1ull << 31) || (uint64_t)K * N * 2 / 32 >= (1ull << 31)) return -1;
  const RegsPlan p = regs_plan(M, N, K, sub, wt == 1);
  if (n_tiles) *n_tiles = p.j;
  if (wavefronts) *wavefronts = p.nw;
  return p.us;
}

void w4a16_regs_workspace(int M, int N, int K, int sub, bool w8, size_t* c_tmp_bytes, size_t* counter_ints) {
  const RegsPlan p = regs_plan(M, N, K, sub, w8);
  *c_tmp_bytes = p.tmp_bytes(N);
  *counter_ints = p.counter_ints(N);
}

int w4a16_regs_launch(const void* a, int64_t lda, const int32_t* b, const void* scales, const int32_t* zeros, const void* bias, void* c,
                      float* c_tmp, int32_t* counters, int M, int N, int K, int sub, bool channelwise, bool w8, int dtype, hipStream_t s) {
  const RegsPlan plan = regs_plan(M, N, K, sub, w8);
  RegsParams p;
  p.a = (const uint16_t*)a;
  p.b = (const v4u*)b;
  p.scales = (const uint16_t*)scales;
  p.zeros = (const uint32_t*)zeros;
  p.bias = (const uint16_t*)bias;
  p.c = (uint16_t*)c;
  p.c_tmp = c_tmp;
  p.counters = counters;
  p.M = M; p.N = N; p.lda = (int)lda;
  p.G = K / 128;
  p.NT = N / 16;
  p.SK = plan.sk;
  p.RB = plan.rb;
  p.ranges = (p.NT + plan.j - 1) / plan.j;
  p.per_xcd = (p.ranges * plan.sk * plan.rb + 7) / 8;
  p.s_stride = channelwise ? 0 : N;
  p.z_stride = channelwise ? 0 : N / 8;
  p.k_mask = 0x000f000fu;
  p.k_ex = dtype == VAQ_BF16 ? 0x43004300u : 0x64006400u;
  const bool bf16 = dtype == VAQ_BF16, zp = zeros != nullptr;
  int rc;
  if (w8) rc = (sub == 1 ? regs_launch_w8 : sub == 2 ? regs_launch_w8_sub2 : regs_launch_w8_sub4)(p, plan.nw, plan.j, plan.mb, bf16, s);
  else rc = (sub == 1 ? regs_launch_w4 : sub == 2 ? regs_launch_w4_sub2 : regs_launch_w4_sub4)(p, plan.nw, plan.j, plan.mb, bf16, zp, s);
  if (rc != VAQ_OK) return rc;
  VAQ_CHECK_LAUNCH("w4a16_gemm(regs)");
  return VAQ_OK;
}

}  // namespace vaq

extern "C" int vaq_w4a16_regs_plan(int64_t size_m, int64_t size_n, int64_t size_k, int sub, int w8, double* plan) {
  using namespace vaq;
  VAQ_CHECK_ARG(size_m > 0 && size_m <= REGS_MAX_M && size_n > 0 && size_n % 64 == 0 && size_k > 0 && size_k % 128 == 0 &&
                    size_n < (1 << 24) && size_k < (1 << 24) && (sub == 1 || sub == 2 || sub == 4) && plan != nullptr,
                "w4a16_regs_plan: bad arguments");
  const RegsPlan p = regs_plan((int)size_m, (int)size_n, (int)size_k, sub, w8 != 0);
  const double out[5] = {(double)p.j, (double)p.mb, (double)p.nw, (double)p.sk, p.us};
  for (int i = 0; i < 5; ++i) plan[i] = out[i];
  double other = -1;
  plan[6] = w4a16_takes_regs((int)size_m, (int)size_n, (int)size_k, sub, w8 != 0 ? 1 : 0, &other) ? 1 : 0;
  plan[5] = other;
  return VAQ_OK;
}
