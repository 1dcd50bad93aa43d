// Which workgroup of a launch computes what: the functions that the kernels call, on the host, against plain divisions.  Over grids of tile counts, parts of K and rows, every
// (tile, part of K) and every (range, part of K, block of rows) is taken once, with the k-tiles that plain division gives.  An argument plants a mistake: 1 in the number for
// bands of tiles, 2 in that for copies, 3 in that for blocks of rows of the FP8 kernel, 4 in that for parts of K.
//
// Build:  hipcc --offload-host-only -O1 -std=c++17 -I vllm_amd/csrc launch_arguments_check.hip -o launch_arguments_check
#include "fp8_regs_kernel.h"
#include "w4a16_regs_kernel.h"

#include <stdio.h>
#include <stdlib.h>

#include <vector>

using namespace vaq;

static long bad = 0, checked = 0;
static void check(bool ok, const char* what, long a, long b, long c, long d) {
  ++checked;
  if (!ok && ++bad < 20) printf("%s: %ld %ld %ld %ld\n", what, a, b, c, d);
}

struct Split {
  int SK, tail_first;
  TileSplitMagic split_magic;
};

static void tiles(int tiles_m, int tiles_n, int sk, int tail_first, int plant) {
  const int all = tiles_m * tiles_n;
  TileGrid g = tile_grid(tiles_m, tiles_n, sk, tail_first);
  if (plant == 1) g.band_magic = g.band_magic / 2;
  Split p{sk, tail_first, tile_split_magic(all, sk, tail_first)};
  if (plant == 4) p.split_magic.sk -= p.split_magic.sk / 8;
  const int gx = tail_first > 0 ? tail_first + (all - tail_first) * sk : all, gy = tail_first > 0 ? 1 : sk;
  std::vector<int> seen((size_t)all * sk, 0), unit((size_t)all, -1);
  for (int y = 0; y < gy; ++y)
    for (int x = 0; x < gx; ++x) {
      const TileSlot s = tile_slot(g, p, x, y);
      const bool there = s.tm >= 0 && s.tm < tiles_m && s.tn >= 0 && s.tn < tiles_n && s.split >= 0 && s.split < s.nsplit && s.nsplit <= sk && s.unit >= 0 && s.unit < s.units;
      check(there, "slot", x, y, s.tm, s.tn);
      if (!there) continue;
      const bool whole = tail_first > 0 && s.pos < tail_first;
      check(s.nsplit == (whole ? 1 : sk) && s.units == all - (tail_first > 0 ? tail_first : 0), "parts", x, y, s.nsplit, s.units);
      const int tile = s.tm * tiles_n + s.tn;
      ++seen[(size_t)tile * sk + s.split];
      if (whole) for (int i = 1; i < sk; ++i) ++seen[(size_t)tile * sk + i];
      else if (unit[s.unit] < 0) unit[s.unit] = tile;
      else check(unit[s.unit] == tile, "unit", x, y, s.unit, tile);
      // bands of four tile rows, column by column
      const int band = s.pos / (TILE_BAND * tiles_n), in = s.pos % (TILE_BAND * tiles_n), high = tiles_m - band * TILE_BAND < TILE_BAND ? tiles_m - band * TILE_BAND : TILE_BAND;
      check(s.tm == band * TILE_BAND + in % high && s.tn == in / high, "order", s.pos, s.tm, s.tn, high);
      for (int steps : {1, 2, 7, 32, 111, 448, 5000, 262143})
        for (int i = 0; i <= s.nsplit; ++i) check(tile_part(p, s, steps, i) == (int)((int64_t)steps * i / s.nsplit), "part of K", steps, i, s.nsplit, tile_part(p, s, steps, i));
    }
  for (size_t i = 0; i < seen.size(); ++i) check(seen[i] == 1, "taken", tiles_m, tiles_n, (long)i, seen[i]);
}

static void registers(int M, int mb, int SK, int NT, int J, int G, int plant) {
  RegsParams p = {};
  p.M = M, p.SK = SK, p.RB = (M + mb * 16 - 1) / (mb * 16), p.NT = NT, p.ranges = (NT + J - 1) / J, p.G = G;
  p.per_xcd = (p.ranges * SK * p.RB + 7) / 8;
  const KernelHead h = regs_head(p);
  const uint32_t counts = h.b[1], ranges = h.b[2], per_xcd = h.b[3], magic = plant == 2 ? h.c[1] - h.c[1] / 16 : h.c[1];
  check((int)(counts & 0x1ff) == M && (int)(counts >> 9 & 0xf) == SK && (int)(counts >> 13 & 0x1f) == p.RB && (int)ranges == p.ranges, "counts", M, SK, p.RB, (long)counts);
  std::vector<int> seen((size_t)p.ranges * SK * p.RB, 0);
  for (uint32_t block = 0; block < per_xcd * 8; ++block) {
    const uint32_t unit = regs_place(block, per_xcd);
    if (unit >= ranges * (uint32_t)(SK * p.RB)) continue;
    const RegsUnit u = regs_unit(unit, counts, magic, (uint32_t)G);
    const bool there = (int)u.range < p.ranges && (int)u.sk < SK && (int)u.rb < p.RB;
    check(there, "range", block, u.range, u.sk, u.rb);
    if (!there) continue;
    ++seen[((size_t)u.range * SK + u.sk) * p.RB + u.rb];
    check((int64_t)u.g_lo == (int64_t)G * u.sk / SK && (int64_t)u.g_hi == (int64_t)G * (u.sk + 1) / SK, "k-tiles", G, u.sk, u.g_lo, u.g_hi);
  }
  for (size_t i = 0; i < seen.size(); ++i) check(seen[i] == 1, "taken", M, SK, (long)i, seen[i]);
}

static void fp8(int RB, int ranges, int plant) {
  const uint32_t per_xcd = ((uint32_t)ranges * RB + 7) / 8, magic = fp8_regs_magic((uint32_t)RB) - (plant == 3 ? fp8_regs_magic((uint32_t)RB) / 16 : 0);
  std::vector<int> seen((size_t)ranges * RB, 0);
  for (uint32_t block = 0; block < per_xcd * 8; ++block) {
    const uint32_t unit = fp8_regs_place(block, per_xcd);
    if (unit >= (uint32_t)ranges * RB) continue;
    const Fp8RegsUnit u = fp8_regs_unit(unit, (uint32_t)RB, magic);
    const bool there = (int)u.range < ranges && (int)u.rb < RB;
    check(there, "fp8 range", block, u.range, u.rb, RB);
    if (there) ++seen[(size_t)u.range * RB + u.rb];
  }
  for (size_t i = 0; i < seen.size(); ++i) check(seen[i] == 1, "fp8 taken", RB, ranges, (long)i, seen[i]);
}

int main(int argc, char** argv) {
  const int plant = argc > 1 ? atoi(argv[1]) : 0;
  for (int m : {1, 2, 3, 4, 5, 6, 7, 8, 9, 13, 16, 31})
    for (int n : {1, 2, 3, 5, 8, 9, 12, 37, 64, 108}) {
      for (int sk : {1, 2, 3, 4, 5, 7, 8, 16}) tiles(m, n, sk, 0, plant);
      for (int sk : {2, 3, 4})
        for (int tail : {1, 7, 8, 64, 256})
          if (tail < m * n) tiles(m, n, sk, tail, plant);
    }
  for (int M : {1, 4, 16, 17, 33, 48, 49, 64, 100, 200, 255, 256})
    for (int mb : {1, 2, 3})
      for (int SK = 1; SK <= 8; ++SK)
        for (int NT : {4, 12, 100, 1792, 9500})
          for (int J : {1, 3, 8}) registers(M, mb, SK, NT, J, SK + M % 113, plant);
  for (int RB = 1; RB <= 16; ++RB)
    for (int ranges : {1, 2, 7, 64, 1000, 37501}) fp8(RB, ranges, plant);
  // the largest numbers of units: quotients at the ends
  for (uint32_t copies = 2; copies <= 128; ++copies)
    for (uint32_t x : {(1u << 25) - 1, (1u << 25) / copies * copies - 1, (1u << 25) / copies * copies - copies})
      check(mul_high(x, (uint32_t)((1ull << 32) / copies + 1)) == x / copies, "copies", x, copies, 0, 0);
  for (uint32_t d : {1u, 2u, 3u, 5u, 7u, 255u, 9504u, 65535u, 65536u, 1u << 20, (1u << 31) - 1, 1u << 31})
    for (uint32_t q : {0u, 1u, 2u, 0xffffffffu / d - (d > 1 ? 1 : 0), 0xffffffffu / d})
      for (uint64_t x : {(uint64_t)q * d, (uint64_t)q * d + d - 1, (uint64_t)q * d + (d > 1)})
        if (x < (1ull << 32)) check(div_by((uint32_t)x, d, div_magic(d)) == (uint32_t)x / d, "quotient", (long)x, d, 0, 0);
  printf("checked=%ld mismatches=%ld\n", checked, bad);
  return bad != 0;
}
