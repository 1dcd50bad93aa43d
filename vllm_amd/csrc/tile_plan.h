// Choice of the tile shape and K split of a tile GEMM: every plan of a problem is priced by a formula whose constants were
// fitted to timings, and the cheapest one is taken.
#pragma once
#include <math.h>
#include <stdint.h>

namespace vaq {

// What a launch of one tile shape costs, in us: a workgroup takes `base` plus, per 64-element (FP8: 64-byte) step of K,
// `step` + `load` * (workgroups per compute unit that run beside it, at most `slots`) + `shared` where two share a
// compute unit; `out` per MB of 16-bit output.
struct TileShape {
  int id, bm, bn, nw, slots;
  double base, step, load, shared, out;
};
// Per MB of weights that come from memory; of a K split: fixed, per part, per MB of all partial tiles (written and read by the
// device) and per MB of one tile's (read by the workgroup that sums them).
struct TileCosts {
  double weight_mb, handover, part, handover_mb, sum_mb;
};

struct TilePlan {
  int id = -1, sk = 1, bm = 0, bn = 0, nw = 0;
  int64_t tiles = 0;
  int64_t tail_first = 0;      // > 0: only the tiles from this position on are split (tile_handover.h)
  int64_t extra_tiles = 0;     // split K: the tiles of a tile row past M that runs beside the real ones (FP8)
  double us = -1;
  double us_strips = -1;       // W4A16: of the cheapest plan without the 256 x 256 tiles of w4a16_tile256_kernel.h
  // scratch of the K split: partial tiles and arrival counters of the tiles that are split
  int64_t split_tiles() const { return sk > 1 ? tiles + extra_tiles - tail_first : 0; }
  int64_t tmp_bytes() const { return (int64_t)sk * split_tiles() * bm * bn * 4; }
  int64_t counter_ints() const { return split_tiles() * nw; }
};

// Predicted time of `tiles` tiles in `sk` parts of K each, or (tail_first > 0) of the tiles from tail_first on in parts
// that make one round, beside whole rounds of the others.
inline double tile_plan_us(const TileShape& t, const TileCosts& c, int64_t M, int64_t N, double weight_bytes, int64_t tiles, int sk,
                           int64_t tail_first, double steps, int64_t cus) {
  const int64_t split_tiles = tail_first > 0 ? tiles - tail_first : tiles, cap = cus * t.slots;
  const int64_t rounds = tail_first > 0 ? tail_first / cus : tiles * sk / cap;
  const double rest = (double)(tail_first > 0 ? split_tiles * sk : tiles * sk % cap) / (double)cus;
  const double part = steps / sk, whole = tail_first > 0 ? steps : part;
  double us = (double)rounds * (t.base + whole * (t.step + t.load * t.slots + (t.slots > 1 ? t.shared : 0)));
  if (rest > 0) us += t.base + part * (t.step + t.load * rest + (rest > 1 ? t.shared : 0));
  const double mem = c.weight_mb * 1e-6 * weight_bytes;
  us = sqrt(sqrt(us * us * us * us + mem * mem * mem * mem)) + 2.0 + t.out * 2e-6 * (double)M * (double)N;
  if (sk > 1) us += c.handover + sk * (c.part + 4e-6 * (double)(t.bm * t.bn) * (c.handover_mb * (double)split_tiles + c.sum_mb));
  return us;
}

// Prices one more plan and keeps it if it is the cheapest so far.  `most_scratch`: plans that need more are left out.
inline void consider_tile_plan(TilePlan& best, const TileShape& t, const TileCosts& c, int64_t M, int64_t N, double weight_bytes,
                               int64_t tiles, int sk, int64_t tail_first, double steps, int64_t cus, int64_t most_scratch) {
  const int64_t scratch = sk > 1 ? (int64_t)sk * (tiles - tail_first) * t.bm * t.bn * 4 : 0;
  if (scratch >= most_scratch) return;
  const double us = tile_plan_us(t, c, M, N, weight_bytes, tiles, sk, tail_first, steps, cus);
  if (best.us >= 0 && us >= best.us) return;
  best.us = us;
  best.id = t.id;
  best.bm = t.bm; best.bn = t.bn; best.nw = t.nw;
  best.tiles = tiles;
  best.sk = sk;
  best.tail_first = tail_first;
}

// A small table of finished plans, one per thread, replaced on collision: weighing the plans of a problem takes 2 us of host
// time.  (Calls that force a part of the plan neither read nor fill it.)  The key's low bits, and those from bit 18 on, move the
// entry: a call that asks for the plans of several formats or kernels of its problem never has them replace one another.
template <class Plan>
struct PlanTable {
  struct Entry {
    int m = -1, n = 0, k = 0, key = 0;
    Plan plan;
  };
  Entry entry[256];
  template <class Make>
  const Plan& get(int m, int n, int k, int key, Make make) {
    const uint32_t at = ((uint32_t)m * 2654435761u ^ (uint32_t)n * 2246822519u ^ (uint32_t)k * 3266489917u) >> 24;
    Entry& e = entry[(at + (uint32_t)key + 8u * ((uint32_t)key >> 18)) & 255];
    if (e.m != m || e.n != n || e.k != k || e.key != key) {
      e.plan = make();
      e.m = m; e.n = n; e.k = k; e.key = key;
    }
    return e.plan;
  }
};
using TilePlanTable = PlanTable<TilePlan>;

}  // namespace vaq
