// Tile GEMMs whose K range is split over workgroups: which workgroup of a launch computes which (tile, K part), and
// how the K parts of a tile become one result.
#pragma once
#include "vaq_common.h"

namespace vaq {

// The (tile, K part) of a workgroup.  Two launch forms:
//  * every tile in `sk` parts: grid (tiles, sk), the part is blockIdx.y;
//  * only the tiles from `tail_first` on (in the order the workgroups take tiles) in `sk` parts, the ones before it whole:
//    grid (tail_first + (tiles - tail_first) * sk).  For tile counts that end in a partly filled round of workgroups:
//    the whole tiles fill the full rounds, the parts of the others fill the last one.
// Consecutive workgroup ids land on different XCDs (round-robin over 8); each XCD gets one contiguous range of tile
// positions (of the whole tiles and of the split ones separately), so that the tiles resident on an XCD are neighbours
// and share operand rows in its L2.  `pos` is the position in tile order, `unit` = the tile's index among the split
// tiles (scratch and counters are laid out by it).
struct TileSlot {
  int pos, split, nsplit, unit, units;
  int tm, tn;      // tile row and column
};

// Integer divisions are emulated in some 30 instructions (64-bit ones in more than 100), and a workgroup that finds its tile by them has gone through
// 600 instructions, fetched cold, before its first request.  x / d = mul_high(x, div_magic(d)), which is at most one short, for any x.  (What follows is
// callable on the host for its test.)
inline uint32_t div_magic(uint32_t d) { return d <= 1 ? 0xffffffffu : (uint32_t)((1ull << 32) / d); }
__host__ __device__ inline uint32_t div_by(uint32_t x, uint32_t d, uint32_t magic) {
  const uint32_t q = mul_high(x, magic);
  return x - q * d >= d ? q + 1 : q;
}

// What a workgroup needs to find its tile, made on the host; in the head of the kernels' arguments (vaq_common.h).
struct TileGrid {
  uint32_t n, m;             // tile columns and rows
  uint32_t band_magic;       // of a band's tiles
  uint32_t per8;             // tiles per XCD where that is a whole number, else 0
  uint32_t flags;            // K parts (12 bits), tail_first > 0, free bits of the kernel's own from 16 on
  __host__ __device__ TileGrid rows(uint32_t tile_rows) const { return TileGrid{n, tile_rows, band_magic, per8, flags}; }
};
constexpr int TILE_BAND = 4;      // tiles are handed out in bands of so many tile rows (2 .. 16 measured: 4 is 1-3 % ahead of 8 on the large shapes)
inline TileGrid tile_grid(int64_t tiles_m, int64_t tiles_n, int sk, int tail_first) {
  const int64_t tiles = tiles_m * tiles_n;
  return TileGrid{(uint32_t)tiles_n, (uint32_t)tiles_m, div_magic((uint32_t)(TILE_BAND * tiles_n)), tiles % 8 == 0 ? (uint32_t)(tiles / 8) : 0u,
                  (uint32_t)sk | (tail_first > 0 ? 1u << 12 : 0u)};
}
// The rest of what a launch with K parts needs, in the parameters of the kernels: SK, tail_first and
struct TileSplitMagic {
  uint32_t sk, rest;      // of the K parts, of the tiles from tail_first on
};
inline TileSplitMagic tile_split_magic(int64_t tiles, int sk, int tail_first) { return TileSplitMagic{div_magic((uint32_t)sk), div_magic((uint32_t)(tiles - tail_first))}; }

// Where K part i of `steps` steps begins.
template <class Params>
__host__ __device__ inline int tile_part(const Params& p, const TileSlot& sl, int steps, int i) {
  if (i >= sl.nsplit) return steps;
  return i == 0 ? 0 : (int)div_by((uint32_t)steps * (uint32_t)i, (uint32_t)sl.nsplit, p.split_magic.sk);
}

template <class Params>
__host__ __device__ inline TileSlot tile_slot_of(const TileGrid& g, const Params& p, int b, int block_y) {
  TileSlot r;
  if (g.flags >> 12 & 1u) {
    const int tail_first = p.tail_first, sk = p.SK, tiles = (int)(g.m * g.n);
    const int rest = tiles - tail_first;
    if (b < tail_first) {
      if (tail_first % 8 == 0) b = (b & 7) * (tail_first / 8) + (b >> 3);
      r.pos = b;
      r.split = 0;
      r.nsplit = 1;
      r.unit = 0;
    } else {
      int q = b - tail_first;
      r.split = (int)div_by((uint32_t)q, (uint32_t)rest, p.split_magic.rest);
      q -= r.split * rest;
      if (rest % 8 == 0 && tail_first % 8 == 0) q = (q & 7) * (rest / 8) + (q >> 3);
      r.pos = tail_first + q;
      r.nsplit = sk;
      r.unit = q;
    }
    r.units = rest;
    return r;
  }
  if (g.per8 > 0) b = (b & 7) * (int)g.per8 + (b >> 3);
  r.pos = b;
  r.split = block_y;
  r.nsplit = (int)(g.flags & 0xfffu);
  r.unit = b;
  r.units = (int)(g.m * g.n);
  return r;
}
// ... and its tile: the tiles resident on one XCD share activation rows and weight columns in its L2.
template <class Params>
__host__ __device__ inline TileSlot tile_slot(const TileGrid& g, const Params& p, int block_x, int block_y) {
  TileSlot r = tile_slot_of(g, p, block_x, block_y);
  const uint32_t in_band = TILE_BAND * g.n, band = div_by((uint32_t)r.pos, in_band, g.band_magic);
  const uint32_t first_m = band * TILE_BAND, tin = (uint32_t)r.pos - band * in_band;
  const uint32_t high = g.m - first_m < TILE_BAND ? g.m - first_m : (uint32_t)TILE_BAND;
  const uint32_t tn = div_by(tin, high, high == 4 ? 0x40000000u : high == 3 ? 0x55555555u : high == 2 ? 0x80000000u : 0xffffffffu);
  r.tm = (int)(first_m + tin - tn * high);
  r.tn = (int)tn;
  return r;
}
template <class Params>
__device__ inline TileSlot tile_slot(const TileGrid& g, const Params& p) { return tile_slot(g, p, (int)blockIdx.x, (int)blockIdx.y); }

// Hand-over of partial tiles.  Each wavefront owns WMB x WNB accumulator blocks of its workgroup's tile and one arrival
// counter per (split tile, wavefront) in the caller's zeroed `counters`.  Every wavefront stores its partial blocks
// (16-byte buffer stores with the sc1 cache-policy bit: device scope, written through to and read from memory that all
// XCDs share -- each XCD has its own L2), waits for their acknowledgement and adds one to the counter; the one that
// finds nsplit - 1 there is the last and sums all parts in split order, starting from zero (the same additions whoever
// is last, so the result does not depend on the order of arrival), and leaves the counter zero.
// (Measured against it on 4096 x 4096 at M = 1024 / 2048 in 2, 4 and 8 parts: a number drawn at the start of the
// kernel that names the summing wavefront, so that it need not store and the others need not be read twice, with a
// bounded wait for the others -- same time in 2 parts, 16-30 % slower in 4 and 8: the wait and its polling cost more
// than the stores they save.  Without any hand-over the same launches take 68 against 83 us in 2 parts of 128 tiles.)
//
// true: this wavefront holds the tile's full sums in `acc` and runs the epilogue; false: it has handed its part over.
template <int WMB, int WNB, int NW>
__device__ inline bool handover_finish(float* c_tmp, int32_t* counters, v16f (&acc)[WMB][WNB], const TileSlot& sl, int wave,
                                       int lane) {
  constexpr int NV4 = WMB * WNB * 4;                       // 16-byte pieces per lane; one unit = NV4 KiB per wavefront
  constexpr int SC1 = 16;
  const int nsplit = sl.nsplit;
  const uint32_t unit = (uint32_t)((sl.unit * NW + wave) * NV4) * 1024u;          // bytes
  const uint32_t split_stride = (uint32_t)sl.units * (uint32_t)(NW * NV4) * 1024u;
  const __amdgpu_buffer_rsrc_t rt = __builtin_amdgcn_make_buffer_rsrc(c_tmp, 0, (int)(split_stride * (uint32_t)nsplit), 0x00020000);
#pragma unroll
  for (int i = 0; i < WMB; ++i)
#pragma unroll
    for (int j = 0; j < WNB; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const v4f v = {acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, v), rt, lane * 16,
                                               (int)(sl.split * split_stride + unit + ((i * WNB + j) * 4 + q) * 1024), SC1);
      }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");        // the part is acknowledged before the counter moves
  int32_t* ctr = counters + (int64_t)sl.unit * NW + wave;
  int old = 0;
  if (lane == 0) old = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  old = __builtin_amdgcn_readfirstlane(old);      // lane 0 holds it; a scalar keeps what depends on it scalar
  if (old != nsplit - 1) return false;
  // CH pieces of two parts in flight at a time (one piece after the other, every load waited for, the last arriver
  // spent NV4 x nsplit memory round trips here); each element is summed in split order, starting from zero.  The last
  // arriver reads its own part back as well: keeping it in registers across this loop instead costs the kernels that
  // run at the register limit more (spills in their main loops) than the reads it saves.
  constexpr int CH = NV4 < 8 ? NV4 : 8;
#pragma unroll
  for (int c0 = 0; c0 < NV4; c0 += CH) {
    v4f sum[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) sum[c] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < nsplit; s0 += 2) {
      const int s1 = s0 + 1 < nsplit ? s0 + 1 : s0;
      v4u r0[CH], r1[CH];
#pragma unroll
      for (int c = 0; c < CH; ++c)
        r0[c] = __builtin_amdgcn_raw_buffer_load_b128(rt, lane * 16, (int)(s0 * split_stride + unit + (c0 + c) * 1024), SC1);
#pragma unroll
      for (int c = 0; c < CH; ++c)
        r1[c] = __builtin_amdgcn_raw_buffer_load_b128(rt, lane * 16, (int)(s1 * split_stride + unit + (c0 + c) * 1024), SC1);
#pragma unroll
      for (int c = 0; c < CH; ++c) sum[c] += __builtin_bit_cast(v4f, r0[c]);
      if (s0 + 1 < nsplit) {
#pragma unroll
        for (int c = 0; c < CH; ++c) sum[c] += __builtin_bit_cast(v4f, r1[c]);
      }
    }
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      const int pc = c0 + c, ij = pc / 4, q = pc % 4;
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[ij / WNB][ij % WNB][4 * q + e] = sum[c][e];
    }
  }
  if (lane == 0) __hip_atomic_store(ctr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

// The same for a wavefront that holds NP 16-byte pieces of the tile's sum per lane (KiB-sized units, one counter per wavefront).
template <int NP, int NW>
__device__ inline bool handover_pieces(float* c_tmp, int32_t* counters, v4f (&part)[NP], const TileSlot& sl, int wave, int lane) {
  constexpr int SC1 = 16;
  const int nsplit = sl.nsplit;
  const uint32_t unit = (uint32_t)((sl.unit * NW + wave) * NP) * 1024u;          // bytes
  const uint32_t split_stride = (uint32_t)sl.units * (uint32_t)(NW * NP) * 1024u;
  const __amdgpu_buffer_rsrc_t rt = __builtin_amdgcn_make_buffer_rsrc(c_tmp, 0, (int)(split_stride * (uint32_t)nsplit), 0x00020000);
#pragma unroll
  for (int c = 0; c < NP; ++c)
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, part[c]), rt, lane * 16, (int)(sl.split * split_stride + unit + c * 1024), SC1);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");        // the part is acknowledged before the counter moves
  int32_t* ctr = counters + (int64_t)sl.unit * NW + wave;
  int old = 0;
  if (lane == 0) old = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  old = __builtin_amdgcn_readfirstlane(old);
  if (old != nsplit - 1) return false;
#pragma unroll
  for (int c = 0; c < NP; ++c) part[c] = v4f{0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < nsplit; s0 += 2) {
    const int s1 = s0 + 1 < nsplit ? s0 + 1 : s0;
    v4u r0[NP], r1[NP];
#pragma unroll
    for (int c = 0; c < NP; ++c) r0[c] = __builtin_amdgcn_raw_buffer_load_b128(rt, lane * 16, (int)(s0 * split_stride + unit + c * 1024), SC1);
#pragma unroll
    for (int c = 0; c < NP; ++c) r1[c] = __builtin_amdgcn_raw_buffer_load_b128(rt, lane * 16, (int)(s1 * split_stride + unit + c * 1024), SC1);
#pragma unroll
    for (int c = 0; c < NP; ++c) part[c] += __builtin_bit_cast(v4f, r0[c]);
    if (s0 + 1 < nsplit) {
#pragma unroll
      for (int c = 0; c < NP; ++c) part[c] += __builtin_bit_cast(v4f, r1[c]);
    }
  }
  if (lane == 0) __hip_atomic_store(ctr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return true;
}

// The same in three steps, for a wavefront whose NP pieces do not all fit its registers a second time: everybody gives its part away (true: the last one), the last one
// takes CH pieces of the sum at a time and, when it has them all, leaves the counter zero.
template <int NP, int NW>
struct HandoverUnit {
  uint32_t unit, split_stride;
  __amdgpu_buffer_rsrc_t rt;
  __device__ HandoverUnit(float* c_tmp, const TileSlot& sl, int wave) {
    unit = (uint32_t)((sl.unit * NW + wave) * NP) * 1024u;          // bytes
    split_stride = (uint32_t)sl.units * (uint32_t)(NW * NP) * 1024u;
    rt = __builtin_amdgcn_make_buffer_rsrc(c_tmp, 0, (int)(split_stride * (uint32_t)sl.nsplit), 0x00020000);
  }
};
template <int NP, int NW, typename Piece>
__device__ inline bool handover_give(float* c_tmp, int32_t* counters, Piece piece, const TileSlot& sl, int wave, int lane) {
  constexpr int SC1 = 16;
  const HandoverUnit<NP, NW> u(c_tmp, sl, wave);
#pragma unroll
  for (int c = 0; c < NP; ++c)
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, piece(c)), u.rt, lane * 16, (int)(sl.split * u.split_stride + u.unit + c * 1024), SC1);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");        // the part is acknowledged before the counter moves
  int old = 0;
  if (lane == 0) old = __hip_atomic_fetch_add(counters + (int64_t)sl.unit * NW + wave, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return __builtin_amdgcn_readfirstlane(old) == sl.nsplit - 1;
}
template <int CH, int NP, int NW>
__device__ inline void handover_take(float* c_tmp, v4f (&sum)[CH], int c0, const TileSlot& sl, int wave, int lane) {
  constexpr int SC1 = 16;
  const HandoverUnit<NP, NW> u(c_tmp, sl, wave);
#pragma unroll
  for (int c = 0; c < CH; ++c) sum[c] = v4f{0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < sl.nsplit; s0 += 2) {
    const int s1 = s0 + 1 < sl.nsplit ? s0 + 1 : s0;
    v4u r0[CH], r1[CH];
#pragma unroll
    for (int c = 0; c < CH; ++c) r0[c] = __builtin_amdgcn_raw_buffer_load_b128(u.rt, lane * 16, (int)(s0 * u.split_stride + u.unit + (c0 + c) * 1024), SC1);
#pragma unroll
    for (int c = 0; c < CH; ++c) r1[c] = __builtin_amdgcn_raw_buffer_load_b128(u.rt, lane * 16, (int)(s1 * u.split_stride + u.unit + (c0 + c) * 1024), SC1);
#pragma unroll
    for (int c = 0; c < CH; ++c) sum[c] += __builtin_bit_cast(v4f, r0[c]);
    if (s0 + 1 < sl.nsplit) {
#pragma unroll
      for (int c = 0; c < CH; ++c) sum[c] += __builtin_bit_cast(v4f, r1[c]);
    }
  }
}
template <int NW>
__device__ inline void handover_done(int32_t* counters, const TileSlot& sl, int wave, int lane) {
  if (lane == 0) __hip_atomic_store(counters + (int64_t)sl.unit * NW + wave, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace vaq
