// W4A16 tile GEMM for many rows: 256 x 256 tiles, weights dequantised in registers, one wavefront to a SIMD.
//
// Four wavefronts, each a strip of 64 columns (four native 16-column tiles) for all 256 rows: 16 x 4 blocks of v_mfma_f32_16x16x32 results, four registers each, in all 256
// accumulation registers, everything else in 128 .. 184 vector registers (4-bit codes in groups of 128 rows 128 .. 140).
//
//  * Weights: a ring of two quantisation groups (128 rows of K) in registers, requested two groups ahead straight from memory.  A native tile's word is the A
//    operand (rows = n) of one MFMA as it lies; dequantised with scale and zero point exactly like the other tile kernels do (fma(code, s, -z s) rounded
//    once, or the same bits by packed fp16).  No weight passes through LDS, and each is dequantised once per 256 rows.
//  * Activations: 64 k of 256 rows per step, global -> LDS by direct-to-LDS loads, four stages of 32 KiB, the image of the LDS-staged kernel (128-byte
//    rows, two to a 256-byte line, 16-byte chunks XOR-ed with the line number).  A fragment is read once and multiplied with four tiles.
//  * One barrier a step, where the first fragment of the next step is read.
//  * One instruction stream holds everything that goes on between two MFMAs: a wavefront alone on its SIMD issues two vector instructions beside a 16-cycle MFMA
//    at no cost (measured 16.3 / 16.6 / 16.7 / 21.7 / 25.2 cycles an MFMA with 0 .. 4 of them), so the dequantisation of the next word is cut into sixteen steps of
//    at most two, one behind each MFMA, and a scheduling barrier behind each keeps them there.
//
// Why this shape.  At this size the device runs at its power limit (the loop with operands that do not toggle is 1.2 .. 1.3 times faster), so what counts is what an MFMA
// takes beside itself.  Against eight wavefronts of 32-column strips (a fragment per two 16 x 16 or one 32 x 32 MFMA) half the LDS reads; 16 x 16 instead of 32 x 32
// MFMAs half the traffic of the accumulators; every other block of rows goes through the tiles backwards, so that from each MFMA to the next one operand stays.
// Measured in turn, 4096 x 4096 / 4096 x 28672 / 14336 x 4096 at M = 4096, bf16, zero points: eight wavefronts of 32 x 32 MFMAs 118 / 778 / 382 us, of 16 x 16 MFMAs 110 /
// 749 / 361, this 107 / 728 / 346, with the tiles backwards 106 / - / 340.
//
// The MFMAs are written as instructions: of the builtin's result, four registers of the 256, the compiler makes a copy per MFMA.  What it would see to itself is done
// by hand: a weight operand is finished at least two instructions ahead of the MFMA that reads it (hardware asks for two between a vector instruction and an
// MFMA that reads its result; here it is a whole word, and the last tile's is read four MFMAs behind its last step), and the accumulators are read behind
// 32 idle cycles.  (The compiler counts the waits for loads that such an instruction reads.)
#pragma once
#include "w4a16_prefill_kernel.h"

namespace vaq {

template <bool BF16, bool HAS_ZP, int SUBG, bool W8>
__global__ __launch_bounds__(256, 1) void w4a16_tile256_kernel(VAQ_HEAD_ARGS, const PrefillParams rest) {
  TileGrid grid;
  const PrefillParams p = prefill_params(h0, h1, h2, rest, grid);
  using T = F16Traits<BF16>;
  constexpr int NW = 4, BM = 256, TN = 64, BN = TN * NW, NST = 4, PD = 2;
  constexpr int TW = TN / 16, MB = BM / 16;        // tiles of 16 columns of a wavefront's strip, blocks of 16 rows
  constexpr int AHEAD = 4;                         // activation fragments are read so many blocks ahead (eight: level)
  constexpr int TPG = W8 ? 2 : 1;
  constexpr int A_LD = BM * 128 / 1024 / NW;       // direct-to-LDS instructions of a wavefront for a step
  constexpr int STAGE = BM * 128;
  constexpr int KW = TW * TPG + TW / 2 * SUBG * (HAS_ZP ? 2 : 1);      // vector-memory instructions of a group's weights
  constexpr bool HP = !BF16;                       // packed fp16 dequantisation
  constexpr int BB = MB + 1 - AHEAD;               // block of a step's second slice ahead of which its barrier stands
  constexpr int SLOTS = (MB - BB + 3) / 4;         // requests between the barrier and the end of its slice, one in every fourth block
  static_assert(!(W8 && HAS_ZP) && A_LD == 8 && MB % AHEAD == 0, "shape");
  static_assert((NST - 2) * A_LD + KW <= 63, "wait counter range");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds8[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  const TileSlot sl = tile_slot(grid.rows((uint32_t)(p.M + BM - 1) / BM), p);
  const int m0 = sl.tm * BM, n0 = sl.tn * BN;
  // K may be split over workgroups: this one covers the groups [g_lo, g_hi)
  const int g_lo = tile_part(p, sl, p.G, sl.split), g_hi = tile_part(p, sl, p.G, sl.split + 1);
  const int ng = g_hi - g_lo;

  // ---- activations.  Rows past M at the far end of the lanes' offsets, steps past the K part at the end of the scalar offset: either requests nothing
  // (zeros, no traffic) and keeps the wait counts uniform; see w4a16_strip_kernel.h. ----
  const uint32_t a_bytes = ((uint32_t)(p.M - 1) * (uint32_t)p.lda + (uint32_t)p.K) * 2u;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.a), 0, (int)a_bytes, 0x00020000);
  uint32_t voff_a[A_LD];
#pragma unroll
  for (int i = 0; i < A_LD; ++i) {
    const int j = (wave * A_LD + i) * 4 + (lane >> 4);
    const int c16 = (lane & 15) ^ (j & 15);
    const int row = m0 + (wave * A_LD + i) * 8 + 2 * (lane >> 4) + (c16 >> 3);
    voff_a[i] = row < p.M ? ((uint32_t)row * (uint32_t)p.lda) * 2u + (uint32_t)(c16 & 7) * 16u : 0xFFFFFF00u;
  }
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  // step h = 2 * group + half
  auto issue_a = [&](int h, int stage, int from, int to) {
    uint8_t* Ab = lds8 + stage * STAGE;
    const int g = g_lo + (h >> 1);
    const uint32_t so = g < g_hi ? (uint32_t)g * 256u + (uint32_t)(h & 1) * 128u : a_bytes;
#pragma unroll
    for (int i = from; i < to; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(Ab + (wave * A_LD + i) * 1024), 16, (int)voff_a[i], (int)so, 0, 0);
  };

  // ---- weights ----
  const int nt0 = n0 / 16 + wave * TW;
  // (one descriptor over the strip: four leave no scalar registers for the rest)
  const int nt_first = min(nt0, p.NT - 1);         // clamped: columns past N are never stored
  const uint32_t w_tile = (uint32_t)p.G * (TPG * 1024), w_bytes = (uint32_t)(min(nt0 + TW, p.NT) - nt_first) * w_tile;
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc(const_cast<v4u*>(p.b + (int64_t)nt_first * p.G * (TPG * 64)), 0, (int)w_bytes, 0x00020000);
  uint32_t voff_w[TW];
#pragma unroll
  for (int i = 0; i < TW; ++i) voff_w[i] = (uint32_t)lane * 16u + (uint32_t)(min(nt0 + i, p.NT - 1) - nt_first) * w_tile;
  int ncol[TW / 2];                  // this lane's column of each pair of tiles: of the first in even rows of 16 lanes, of the second in odd ones
#pragma unroll
  for (int nb = 0; nb < TW / 2; ++nb) ncol[nb] = min(nt0 + 2 * nb + ((lane >> 4) & 1), p.NT - 1) * 16 + (lane & 15);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.scales), 0, (p.s_stride * (p.G * SUBG - 1) + p.N) * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t rz = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(p.zeros), 0, (p.z_stride * (p.G * SUBG - 1) + p.N / 8) * 4, 0x00020000);
  struct WSet {
    v4u w[TW][TPG];
    uint16_t s[TW / 2][SUBG];
    uint32_t z[TW / 2][SUBG];
  };
  WSet ring[PD];
  // tile t's part of the requests of a group
  auto load_w = [&](WSet& d, int group, int t) {
    const int g = g_lo + group, gc = min(g, g_hi - 1);
    const uint32_t so = g < g_hi ? (uint32_t)g * (TPG * 1024) : w_bytes;      // past the end: zeros, no traffic
#pragma unroll
    for (int b = 0; b < TPG; ++b) d.w[t][b] = __builtin_amdgcn_raw_buffer_load_b128(rw, (int)(voff_w[t] + b * 1024), (int)so, 0);
    if (t & 1) {
      const int nb = t >> 1;
#pragma unroll
      for (int sj = 0; sj < SUBG; ++sj) {
        const int row = gc * SUBG + sj;
        d.s[nb][sj] = __builtin_amdgcn_raw_buffer_load_b16(rs, ncol[nb] * 2, row * p.s_stride * 2, 0);
        if constexpr (HAS_ZP) d.z[nb][sj] = __builtin_amdgcn_raw_buffer_load_b32(rz, (ncol[nb] >> 3) * 4, row * p.z_stride * 4, 0);
        else d.z[nb][sj] = 0u;
      }
    }
  };
  // (a copy that stays one: merged with the ring's register it makes the whole ring change places once a turn, which waits for all of its requests)
  auto moved = [](uint32_t x) {
    uint32_t y;
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("v_mov_b32 %0, %1" : "=&v"(y) : "v"(x));
#else
    y = x;
#endif
    return y;
  };
  // current group: words [tile][j], high and low nibbles of 8-bit codes; scale and -(zero * scale) of the sub-group at hand by tile (floats, or pairs of fp16)
  uint32_t wcur[TW][4], wlo[TW][W8 ? 4 : 1];
  uint32_t s_hold[TW / 2][SUBG], z_hold[TW / 2][SUBG];      // of the current group, beyond the first sub-group
  uint32_t s_of[TW], z_of[TW];
  auto take_words = [&](const WSet& d, int t) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      wcur[t][j] = moved(d.w[t][0][j]);
      if constexpr (W8) wlo[t][j] = moved(d.w[t][TPG - 1][j]);
    }
  };
  auto take_scales = [&](int nb, uint32_t sraw, uint32_t zraw) {
    uint32_t zc = W8 ? 128u : 8u, s, z;
    if constexpr (HAS_ZP) zc = (zraw >> ((lane & 7) * 4)) & 0xFu;
    if constexpr (HP) {
      const uint32_t zb = 0xE400u | zc;
      s = sraw | (sraw << 16);
      z = zb | (zb << 16);
    } else {
      const float sv = T::to_float((uint16_t)sraw);
      s = __float_as_uint(sv);
      z = __float_as_uint(-((float)zc * sv));
    }
    const auto sv = __builtin_amdgcn_permlane16_swap(s, s, false, false);
    const auto zv = __builtin_amdgcn_permlane16_swap(z, z, false, false);
    s_of[2 * nb] = sv[0];
    s_of[2 * nb + 1] = sv[1];
    z_of[2 * nb] = zv[0];
    z_of[2 * nb + 1] = zv[1];
  };
  auto take_group_scales = [&](const WSet& d, int nb) {
    take_scales(nb, d.s[nb][0], d.z[nb][0]);
    if constexpr (SUBG > 1) {
#pragma unroll
      for (int sj = 1; sj < SUBG; ++sj) {
        s_hold[nb][sj] = moved(d.s[nb][sj]);
        if constexpr (HAS_ZP) z_hold[nb][sj] = moved(d.z[nb][sj]);
        else z_hold[nb][sj] = 0u;
      }
    }
  };

  v4f acc[MB][TW];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int t = 0; t < TW; ++t) {
      acc[i][t] = v4f{0.f, 0.f, 0.f, 0.f};
#ifdef __HIP_DEVICE_COMPILE__
      asm volatile("" : "+a"(acc[i][t]));
#endif
    }
  auto multiply = [&](int i, int t, v4u w, v4u a) {
#ifdef __HIP_DEVICE_COMPILE__
    if constexpr (BF16) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][t]) : "v"(w), "v"(a));
    else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc[i][t]) : "v"(w), "v"(a));
#endif
  };

  // operand reads of slice jj (= word) of a step: row lane & 15 of a block, 16-byte chunk 4 jj + (lane >> 4) of its 128-byte row; odd blocks lie
  // eight lines further on
  uint32_t coff[2][2];
#pragma unroll
  for (int jj = 0; jj < 2; ++jj)
#pragma unroll
    for (int odd = 0; odd < 2; ++odd) {
      const int chunk = 4 * jj + (lane >> 4), line = 8 * odd + ((lane & 15) >> 1);
      coff[jj][odd] = (uint32_t)(line * 256 + ((((lane & 1) * 8 + chunk) ^ line) * 16));
    }
  v4u af[AHEAD];
  v4u wf[2][TW];
  auto read_a = [&](const uint8_t* stage, int jj, int block) {
    af[block % AHEAD] = *reinterpret_cast<const v4u*>(stage + (block >> 1) * 4096 + coff[jj][block & 1]);
  };

  // the steps of the dequantisation of one word of tile t, one to two vector instructions each, between two MFMAs
  typedef float v2f __attribute__((ext_vector_type(2)));
  struct {
    uint32_t x;
    v2f lo, hi;
    float l, h;
  } d;
  auto dequant_step = [&](v4u& out, int t, int j, int s) {
    const float sf = __uint_as_float(s_of[t]), zf = __uint_as_float(z_of[t]);
    if constexpr (HP) {
      const int q = s >> 2;
      if constexpr (W8) {
        if ((s & 3) == 1) d.x = (q & 1) ? (wcur[t][j] & 0xf0f0f0f0u) | ((wlo[t][j] >> 4) & 0x0f0f0f0fu) : ((wcur[t][j] << 4) & 0xf0f0f0f0u) | (wlo[t][j] & 0x0f0f0f0fu);
        if ((s & 3) == 2) d.x = q < 2 ? (d.x & 0x00ff00ffu) | 0x64006400u : __builtin_amdgcn_perm(0x64646464u, d.x, 0x04030401u);
      } else {
        if ((s & 3) == 1) d.x = ((wcur[t][j] >> (4 * q)) & 0x000f000fu) | 0x64006400u;
      }
      if ((s & 3) == 3) out[q] = __builtin_bit_cast(uint32_t, (__builtin_bit_cast(v2h, d.x) + __builtin_bit_cast(v2h, z_of[t])) * __builtin_bit_cast(v2h, s_of[t]));
    } else if constexpr (W8) {
      const int q = s < 4 ? 0 : s < 8 ? 2 : s < 12 ? 1 : 3;
      if (s == 0) d.x = ((wcur[t][j] & 0x0f0f0f0fu) << 4) | (wlo[t][j] & 0x0f0f0f0fu);
      if (s == 8) d.x = (wcur[t][j] & 0xf0f0f0f0u) | ((wlo[t][j] >> 4) & 0x0f0f0f0fu);
      if ((s & 3) == 1) {
        d.l = q >> 1 ? cvt_ubyte<1>(d.x) : cvt_ubyte<0>(d.x);
        d.h = q >> 1 ? cvt_ubyte<3>(d.x) : cvt_ubyte<2>(d.x);
      }
      if ((s & 3) == 2) {
        d.l = fmaf(d.l, sf, zf);
        d.h = fmaf(d.h, sf, zf);
      }
      if ((s & 3) == 3) out[q] = pack2<BF16>(d.l, d.h);
    } else {
      if (s == 0) d.x = wcur[t][j] & 0x0f0f0f0fu;
      if (s == 1) d.lo = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(d.x, 512.0f, false);
      if (s == 2) d.hi = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(d.x, 512.0f, true);
      if (s == 3) { d.l = fmaf(d.lo[0], sf, zf); d.h = fmaf(d.hi[0], sf, zf); }
      if (s == 4) out[0] = pack2<BF16>(d.l, d.h);
      if (s == 5) { d.l = fmaf(d.lo[1], sf, zf); d.h = fmaf(d.hi[1], sf, zf); }
      if (s == 6) { out[2] = pack2<BF16>(d.l, d.h); d.x = wcur[t][j] >> 4; }
      if (s == 7) d.x &= 0x0f0f0f0fu;
      if (s == 8) d.lo = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(d.x, 512.0f, false);
      if (s == 9) d.hi = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(d.x, 512.0f, true);
      if (s == 10) { d.l = fmaf(d.lo[0], sf, zf); d.h = fmaf(d.hi[0], sf, zf); }
      if (s == 11) out[1] = pack2<BF16>(d.l, d.h);
      if (s == 13) { d.l = fmaf(d.lo[1], sf, zf); d.h = fmaf(d.hi[1], sf, zf); }
      if (s == 14) out[3] = pack2<BF16>(d.l, d.h);
    }
  };

  // Vector-memory operations retire in issue order.  Where step h's last fragments are read the activations of step h + 1 must have landed; newer than they are
  // those of the NST - 2 steps behind them and the weights of one group.
  constexpr int WAIT = (NST - 2) * A_LD + KW * ((NST - 2) / 2);

  auto nothing = [] {};
  // One k-slice, 32 k: word jj of the step in `here`.  In the shadow of its MFMAs the activation fragments AHEAD blocks on (behind the step's last in the
  // stage `there`, which `arrived` waits for), the dequantisation of word next_j, a fourth of the slice for each tile, and at the end of that fourth what comes
  // next for the tile: its words of the next group, its scales of the next sub-group.
  auto slice = [&](auto jj_c, const uint8_t* here, const uint8_t* there, auto next_j_c, const WSet& nxt, auto arrived, auto request, auto weights) {
    constexpr int jj = decltype(jj_c)::value, next_j = decltype(next_j_c)::value, cbuf = jj, nbuf = jj ^ 1;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int t = 0; t < TW; ++t) {
        const int tt = i / (MB / TW), s = (i % (MB / TW)) * TW + t;
        if (jj == 1 && i == BB && t == 0) arrived();
        const int tx = i & 1 ? TW - 1 - t : t;
        multiply(i, tx, wf[cbuf][tx], af[i % AHEAD]);
        if (t == 0) {
          const int b = i - 1 + AHEAD;
          if (b < MB) read_a(here, jj, b);
          else read_a(jj == 0 ? here : there, jj ^ 1, b - MB);
        }
        dequant_step(wf[nbuf][tt], tt, next_j, s);
        if (s == 13) weights(tt);
        if (s == 14) request(tt);
        if (s == 15 && next_j == 3) take_words(nxt, tt);
        if (s == 15 && (tt & 1)) {
          if (next_j == 3) take_group_scales(nxt, tt >> 1);
          else if (SUBG > 1 && (next_j + 1) * SUBG % 4 == 0) take_scales(tt >> 1, s_hold[tt >> 1][(next_j + 1) * SUBG / 4 % SUBG], z_hold[tt >> 1][(next_j + 1) * SUBG / 4 % SUBG]);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
  };
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
  using C2 = std::integral_constant<int, 2>;
  using C3 = std::integral_constant<int, 3>;

  // ---- prologue: the requests of the first NST steps (of the last as many as the loop makes behind a barrier) and PD groups, in the loop's order ----
  auto keep_order = [] { asm volatile("" ::: "memory"); __builtin_amdgcn_sched_barrier(0); };
  issue_a(0, 0, 0, A_LD);
#pragma unroll
  for (int t = 0; t < TW; ++t) load_w(ring[0], 0, t);
  keep_order();
  issue_a(1, 1, 0, A_LD);
  keep_order();
#pragma unroll
  for (int t = 0; t < TW; ++t) load_w(ring[1], 1, t);
  keep_order();
  issue_a(2, 2, 0, A_LD);
  keep_order();
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 2) * A_LD + (PD - 1) * KW) : "memory");
#pragma unroll
  for (int t = 0; t < TW; ++t) take_words(ring[0], t);
#pragma unroll
  for (int nb = 0; nb < TW / 2; ++nb) take_group_scales(ring[0], nb);
  issue_a(NST - 1, NST - 1, 0, SLOTS);
#pragma unroll
  for (int t = 0; t < TW; ++t)
#pragma unroll
    for (int s = 0; s < 16; ++s) dequant_step(wf[0][t], t, 0, s);
  // (scales for word 1)
  if constexpr (SUBG == 4) {
#pragma unroll
    for (int nb = 0; nb < TW / 2; ++nb) take_scales(nb, s_hold[nb][1], z_hold[nb][1]);
  }
  asm volatile("s_nop 4\n\ts_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < AHEAD - 1; ++i) read_a(lds8, 0, i);

  int cur = 0;
  auto next_stage = [](int x) { return x + 1 == NST ? 0 : x + 1; };
  // a group: its two steps; `fly` = ring slot that is being refilled, `nxt` = the next group's (`last_c`: the group behind the loop requests no more weights)
  auto round = [&](int r, WSet& fly, WSet& nxt, auto last_c) {
    constexpr bool last = decltype(last_c)::value;
    auto no_weights = [](int) {};
    auto weights = [&](int t) {
      if constexpr (!last) load_w(fly, r + PD, t);
    };
    auto step_end = [&] {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(last ? (NST - 2) * A_LD : WAIT) : "memory");
    };
    const uint8_t* A0 = lds8 + cur * STAGE;
    const int s1 = next_stage(cur), s2 = next_stage(s1), sp = cur == 0 ? NST - 1 : cur - 1;
    const uint8_t* A1 = lds8 + s1 * STAGE;
    const uint8_t* A2 = lds8 + s2 * STAGE;
    const int ha = 2 * r - 1 + NST;
    auto place = [&](auto k_c) {      // slice k's requests
      return [&](int tt) {
        const int x = decltype(k_c)::value * 4 + tt + SLOTS;
        issue_a(ha + x / 8, x < 8 ? sp : x < 16 ? cur : s1, x % 8, x % 8 + 1);
      };
    };
    slice(C0{}, A0, A0, C1{}, nxt, nothing, place(C0{}), weights);
    slice(C1{}, A0, A1, C2{}, nxt, step_end, place(C1{}), no_weights);
    slice(C0{}, A1, A1, C3{}, nxt, nothing, place(C2{}), no_weights);
    slice(C1{}, A1, A2, C0{}, nxt, step_end, place(C3{}), no_weights);
    cur = s2;
  };
  using IN_LOOP = std::false_type;
  using BEHIND = std::true_type;
  int r = 0;
  for (; r + PD <= ng; r += PD) {
    round(r, ring[0], ring[1], IN_LOOP{});
    round(r + 1, ring[1], ring[0], IN_LOOP{});
  }
  if (r < ng) round(r, ring[0], ring[1], BEHIND{});
#ifdef __HIP_DEVICE_COMPILE__
  // (the results of the last MFMAs, which the compiler knows nothing of)
  asm volatile("s_nop 15\n\ts_nop 15\n\ts_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int t = 0; t < TW; ++t) asm volatile("" : "+a"(acc[i][t]));
#endif
  __builtin_amdgcn_sched_barrier(0);

  constexpr int PIECES = MB * TW, CH = 8;      // piece = TW * block + tile
  const bool split = sl.nsplit > 1;
  if (split && !handover_give<PIECES, NW>(p.c_tmp, p.counters, [&](int c) { return acc[c / TW][c % TW]; }, sl, wave, lane)) return;

  // ---- bias, rounding, stores: a piece holds 16 columns of row lane & 15 of its block, columns 4 * (lane >> 4) + 0..3 of them in this lane; two
  // neighbouring tiles exchange rows of 16 lanes so that every lane stores 16 bytes, and four lanes the 64 bytes of a row ----
  const int nb0 = n0 + wave * TN, lq = lane >> 4;
  const bool wide = ((uintptr_t)p.c & 15) == 0;
#pragma unroll
  for (int c0 = 0; c0 < PIECES; c0 += CH) {
    v4f sum[CH];
    if (split) handover_take<CH, PIECES, NW>(p.c_tmp, sum, c0, sl, wave, lane);
    else {
#pragma unroll
      for (int c = 0; c < CH; ++c) sum[c] = acc[(c0 + c) / TW][(c0 + c) % TW];
    }
#pragma unroll
    for (int c = 0; c < CH; c += 2) {
      const int pc = c0 + c, mrow = m0 + 16 * (pc / TW) + (lane & 15), nc = nb0 + 16 * (pc % TW);
      if (nc >= p.N) continue;
      v2u pk[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        v4f v = sum[c + x];
        if (p.bias && nc + 16 * x < p.N) {
          const v2u bb = *reinterpret_cast<const v2u*>(p.bias + nc + 16 * x + 4 * lq);
          v[0] += T::to_float((uint16_t)(bb.x & 0xffffu));
          v[1] += T::to_float((uint16_t)(bb.x >> 16));
          v[2] += T::to_float((uint16_t)(bb.y & 0xffffu));
          v[3] += T::to_float((uint16_t)(bb.y >> 16));
        }
        pk[x].x = pack2<BF16>(v[0], v[1]);
        pk[x].y = pack2<BF16>(v[2], v[3]);
      }
      if (mrow >= p.M && !wide) continue;
      uint16_t* row = p.c + (int64_t)mrow * p.N + nc;
      if (wide) {
        const auto s0 = __builtin_amdgcn_permlane16_swap(pk[0].x, pk[1].x, false, false);
        const auto s1 = __builtin_amdgcn_permlane16_swap(pk[0].y, pk[1].y, false, false);
        const int at = 16 * (lq & 1) + 8 * (lq >> 1);
        if (mrow < p.M && nc + at < p.N) *reinterpret_cast<v4u*>(row + at) = v4u{s0[0], s1[0], s0[1], s1[1]};
      } else {
#pragma unroll
        for (int x = 0; x < 2; ++x)
          if (nc + 16 * x < p.N) *reinterpret_cast<v2u*>(row + 16 * x + 4 * lq) = pk[x];
      }
    }
  }
  if (split) handover_done<NW>(p.counters, sl, wave, lane);
}

template <bool BF16, bool HAS_ZP, int SUBG, bool W8>
static int launch_tile256(const PrefillParams& p_in, hipStream_t s) {
  PrefillParams p = p_in;
  constexpr size_t lds = 4 * 256 * 128;
  auto kern = w4a16_tile256_kernel<BF16, HAS_ZP, SUBG, W8>;
  static size_t reserved[VAQ_MAX_DEVICES];
  if (const int rc = reserve_dynamic_lds(reinterpret_cast<const void*>(kern), lds, reserved, "w4a16_gemm(256 x 256)"); rc != VAQ_OK) return rc;
  const int tiles_m = (p.M + 255) / 256, tiles_n = (p.N + 255) / 256, tiles = tiles_m * tiles_n;
  const KernelHead h = prefill_head(p, tile_grid(tiles_m, tiles_n, p.SK, p.tail_first));
  p.split_magic = tile_split_magic(tiles, p.SK, p.tail_first);
  const dim3 grid = p.tail_first > 0 ? dim3(p.tail_first + (tiles - p.tail_first) * p.SK) : dim3(tiles, p.SK);
  hipLaunchKernelGGL(kern, grid, dim3(256), lds, s, h.a, h.b, h.c, p);
  return VAQ_OK;
}

}  // namespace vaq
