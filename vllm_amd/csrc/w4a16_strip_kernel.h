// W4A16 tile GEMM: weight strips dequantised in registers, K groups side by side in a workgroup.
//
// A workgroup of eight wavefronts computes BM = 32 * WMB rows x BN = 32 * WNB * NS columns.  A wavefront owns one strip of 32 * WNB
// columns (pairs of native 16-column tiles) for all BM rows, and one of KG = 8 / NS groups of every KG consecutive quantisation
// groups (128 rows of K each); the KG partial sums of a tile meet in LDS at the end.
//
//  * Weights: a ring of PD groups per wavefront in registers, requested PD rounds ahead straight from memory.  Two neighbouring
//    native tiles become the A operand (rows = n) of v_mfma_f32_32x32x16 after one v_permlane16_swap per word, dequantised with
//    scale and zero point exactly like the LDS-staged kernel does (fma(code, s, -z s) rounded once), in the shadow of the MFMAs of
//    the slice before.  No weight passes through LDS, and each is dequantised once per tile.
//  * Activations: half a group (64 k) of KG groups x BM rows per step, global -> LDS by direct-to-LDS loads, NST stages, the image
//    of the LDS-staged kernel (128-byte rows, two to a 256-byte line, 16-byte chunks XOR-ed with the line number).
//  * One workgroup barrier per step (64 k of every group), placed in front of the slice in which the next step's fragments are first read.
//
// What it is for: the LDS-staged kernel's K step of 64 is a chain -- barrier, fragment reads, MFMAs, weight writes -- of 0.55 us
// whatever the tile, so that tens to hundreds of rows ran at a fifth of the matrix core's rate and needed K in many parts, with
// their hand-over, to fill the device.  Here a step is 2 KG times the work per barrier, a split of K over the workgroup's own
// wavefronts replaces most of the split over workgroups, and weights skip the way through LDS.  Cold, us, the fastest plan of the
// LDS-staged shapes -> of these: 4096 x 6144 at M = 96 / 200 / 333 / 512 / 1024 19.1 / 27.0 / 33.1 / 40.1 / 62.8 -> 14.7 / 21.5 / 27.3
// / 32.7 / 54.4, 4096 x 4096 at M = 256 / 512 / 2048 21.2 / 31.0 / 73.7 -> 16.8 / 25.3 / 63.1, 4096 x 28672 at M = 64 / 128 / 256
// 34.1 / 46.2 / 72.0 -> 26.9 / 37.6 / 59.9, 14336 x 4096 at M = 64 / 512 26.0 / 75.4 -> 21.2 / 66.1.
// What bounds it now (timing-only builds of 4096 x 6144 at M = 512 on 128 x 128 tiles, 34 us): 8 us for launch, first loads, partial
// sums and stores; the K loop's MFMAs alone 13.7 us, with fragment reads and dequantisation 18 us (up to 64 rows the 19 VALU
// instructions per 8 weights take longer than the MFMAs that hide them); operands that toggle 5 us (power); the rest is the memory
// traffic beside it (all operands from memory without arithmetic: 13 us).  Not kept: all requests of a step at once behind the
// barrier (+1 us), more stages (level).
#pragma once
#include "w4a16_prefill_kernel.h"

namespace vaq {

template <int WMB, int WNB, int NS>
constexpr size_t strip_lds_bytes(int nst) {
  constexpr int KG = 8 / NS;
  const size_t stages = (size_t)nst * KG * WMB * 4096, sums = (size_t)(KG - 1) * NS * WMB * WNB * 4096;
  return stages > sums ? stages : sums;
}

// (The smallest strips with zero points of four groups: two workgroups to a compute unit, which 128 registers allow and 130 do not.)
template <bool BF16, int WMB, int WNB, int NS, bool HAS_ZP, int SUBG, bool W8, int NST, int PD>
__global__ __launch_bounds__(512, WMB * WNB == 1 && HAS_ZP && SUBG == 4 ? 4 : 2) void w4a16_strip_kernel(VAQ_HEAD_ARGS, const PrefillParams rest) {
  TileGrid grid;
  const PrefillParams p = prefill_params(h0, h1, h2, rest, grid);
  using T = F16Traits<BF16>;
  constexpr int KG = 8 / NS, BM = 32 * WMB, TN = 32 * WNB, BN = TN * NS, NW = 8;
  constexpr int TW = 2 * WNB;                      // native tiles of a strip
  constexpr int TPG = W8 ? 2 : 1;
  constexpr int A_LD = 4 * WMB / NS;               // direct-to-LDS instructions per wavefront and step
  constexpr int STAGE = KG * BM * 128;             // bytes
  // Activation fragments are read two slices ahead, else one.  8-bit codes: a slice's dequantisation is so long that the two wavefronts of a SIMD rarely overlap, and a read of one
  // slice's length is waited for.  Cold, all groups, of the time with reads one slice ahead: 96 x 128 0.93 .. 0.985 (4096 x 28672 at M = 120, 64-row groups, 70.0 -> 65.4 us), 128 x 128
  // 0.97 .. 1.0, 128 x 256 0.905 .. 0.957 (4096 x 4096 at M = 333 54.5 -> 50.3), 64 x 128 0.94 .. 0.987, but in groups of 32 level; 32 x 128, 64 x 64 and 32 x 64 0.97 .. 1.04.
  // 4-bit codes on 96 x 128 0.98 .. 1.04, on 128 x 128 1.01 .. 1.03.
  constexpr bool DEEP = W8 && WNB == 1 && (WMB >= 3 || (WMB == 2 && NS == 4 && SUBG < 4));
  constexpr int KW = TW * TPG + WNB * SUBG * (HAS_ZP ? 2 : 1);      // vector-memory instructions of one load_w
  constexpr bool HP = !BF16 && SUBG < 4;              // packed fp16 dequantisation (its constants of four sub-groups do not fit the registers)
  static_assert(KG * NS == 8 && (4 * WMB) % NS == 0 && (WMB * WNB * 4) % KG == 0 && !(W8 && HAS_ZP), "strip kernel: shape");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds8[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave / NS, ns = wave % NS;

  const TileSlot sl = tile_slot(grid.rows((uint32_t)(p.M + BM - 1) / BM), p);
  const int m0 = sl.tm * BM, n0 = sl.tn * BN;
  // K may be split over workgroups: this one covers the groups [g_lo, g_hi)
  const int g_lo = tile_part(p, sl, p.G, sl.split), g_hi = tile_part(p, sl, p.G, sl.split + 1);
  const int ng = g_hi - g_lo;
  const int t_full = ng / KG, rem = ng % KG;       // rounds in which all K groups take part; wavefronts of the last one

  // ---- activations: the rows of this wavefront's own K group are loaded by its NS wavefronts ----
  // A descriptor of the rows' own bytes and no more: an operand may be the trailing columns of its storage.  The rows are in the lanes' offsets
  // (up to 4 GiB, checked on the host), those past M at its far end; the scalar offset is the place in K, or all of the extent for a group past the
  // K part (vaq_common.h): either requests nothing (zeros, no traffic) and keeps the wait counts uniform.  (Row tests and a select for
  // every request cost 0.7 % in the mean over 1300 problems of M = 200 .. 4096; rows in the scalar offset, one addition a request, 0.3 % over 3250.)
  const uint32_t a_bytes = ((uint32_t)(p.M - 1) * (uint32_t)p.lda + (uint32_t)p.K) * 2u;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.a), 0, (int)a_bytes, 0x00020000);
  uint32_t voff_a[A_LD];
#pragma unroll
  for (int i = 0; i < A_LD; ++i) {
    const int j = (ns * A_LD + i) * 4 + (lane >> 4);
    const int c16 = (lane & 15) ^ (j & 15);
    const int row = m0 + (ns * A_LD + i) * 8 + 2 * (lane >> 4) + (c16 >> 3);
    voff_a[i] = row < p.M ? ((uint32_t)row * (uint32_t)p.lda) * 2u + (uint32_t)(c16 & 7) * 16u : 0xFFFFFF00u;
  }
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  // step h = 2 * round + half
  auto issue_a = [&](int h, int stage, int from, int to) {
    uint8_t* Ab = lds8 + stage * STAGE + kg * (BM * 128);
    const int g = g_lo + (h >> 1) * KG + kg;
    const uint32_t so = g < g_hi ? (uint32_t)g * 256u + (uint32_t)(h & 1) * 128u : a_bytes;
#pragma unroll
    for (int i = from; i < to; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(Ab + (ns * A_LD + i) * 1024), 16, (int)voff_a[i], (int)so, 0, 0);
  };

  // ---- weights ----
  const int nt0 = n0 / 16 + ns * TW;
  __amdgpu_buffer_rsrc_t rw[TW];
#pragma unroll
  for (int i = 0; i < TW; ++i)       // clamped: columns past N are never stored
    rw[i] = __builtin_amdgcn_make_buffer_rsrc(const_cast<v4u*>(p.b + (int64_t)min(nt0 + i, p.NT - 1) * p.G * (TPG * 64)), 0, g_hi * (TPG * 1024), 0x00020000);
  int ncol[WNB];                     // this lane's column of each 32-column block
#pragma unroll
  for (int nb = 0; nb < WNB; ++nb) ncol[nb] = min(nt0 + 2 * nb + ((lane >> 4) & 1), p.NT - 1) * 16 + (lane & 15);
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.scales), 0, (p.s_stride * (p.G * SUBG - 1) + p.N) * 2, 0x00020000);
  const __amdgpu_buffer_rsrc_t rz = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(p.zeros), 0, (p.z_stride * (p.G * SUBG - 1) + p.N / 8) * 4, 0x00020000);
  struct WSet {
    v4u w[TW][TPG];
    uint16_t s[WNB][SUBG];
    uint32_t z[WNB][SUBG];
  };
  WSet ring[PD];
  // quarter q of the requests of a round (two halves of the tiles, the scales, the zero points)
  auto load_w_q = [&](WSet& d, int round, int q) {
    const int g = g_lo + round * KG + kg, gc = min(g, g_hi - 1);
    const int so = min(g, g_hi) * (TPG * 1024);      // past the end: zeros, no traffic
    if (q < 2) {
#pragma unroll
      for (int i = q * WNB; i < (q + 1) * WNB; ++i)
#pragma unroll
        for (int b = 0; b < TPG; ++b) d.w[i][b] = __builtin_amdgcn_raw_buffer_load_b128(rw[i], lane * 16 + b * 1024, so, 0);
    } else {
#pragma unroll
      for (int nb = 0; nb < WNB; ++nb)
#pragma unroll
        for (int sj = 0; sj < SUBG; ++sj) {
          const int row = gc * SUBG + sj;
          if (q == 2) d.s[nb][sj] = __builtin_amdgcn_raw_buffer_load_b16(rs, ncol[nb] * 2, row * p.s_stride * 2, 0);
          else if constexpr (HAS_ZP) d.z[nb][sj] = __builtin_amdgcn_raw_buffer_load_b32(rz, (ncol[nb] >> 3) * 4, row * p.z_stride * 4, 0);
          else d.z[nb][sj] = 0u;
        }
    }
  };
  auto load_w = [&](WSet& d, int round) {
#pragma unroll
    for (int q = 0; q < 4; ++q) load_w_q(d, round, q);
  };
  // current group: swapped words [block][j][X' / Y'], scale and -(zero * scale) per sub-group
  uint32_t wsw[WNB][4][2], wlo[WNB][W8 ? 4 : 1][2];      // (8-bit codes: high and low nibbles)
  float scur[WNB][SUBG], zcur[WNB][SUBG];
  uint32_t s2cur[WNB][HP ? SUBG : 1], nzb2cur[WNB][HP ? SUBG : 1];
  auto advance_w = [&](const WSet& d) {
#pragma unroll
    for (int nb = 0; nb < WNB; ++nb) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const auto sw = __builtin_amdgcn_permlane16_swap(d.w[2 * nb][0][j], d.w[2 * nb + 1][0][j], false, false);
        wsw[nb][j][0] = sw[0];
        wsw[nb][j][1] = sw[1];
        if constexpr (W8) {
          const auto sv = __builtin_amdgcn_permlane16_swap(d.w[2 * nb][TPG - 1][j], d.w[2 * nb + 1][TPG - 1][j], false, false);
          wlo[nb][j][0] = sv[0];
          wlo[nb][j][1] = sv[1];
        }
      }
#pragma unroll
      for (int sj = 0; sj < SUBG; ++sj) {
        const float sv = T::to_float(d.s[nb][sj]);
        uint32_t zc = W8 ? 128u : 8u;
        if constexpr (HAS_ZP) zc = (d.z[nb][sj] >> ((lane & 7) * 4)) & 0xFu;
        scur[nb][sj] = sv;
        zcur[nb][sj] = -((float)zc * sv);                        // exact: <= 8 + 11 significant bits
        if constexpr (HP) {
          const uint32_t sb = d.s[nb][sj], zb = 0xE400u | zc;    // -(1024 + zero) as fp16 bits
          s2cur[nb][sj] = sb | (sb << 16);
          nzb2cur[nb][sj] = zb | (zb << 16);
        }
      }
    }
  };
  // register q (0..3) of the 16-bit A operand of slice (j, xy) for block nb
  auto dequant_q = [&](int nb, int j, int xy, int q) -> uint32_t {
    const int sj = (j * SUBG) >> 2;
    if constexpr (W8 && HP) return dequant_pair8_h(wsw[nb][j][xy], wlo[nb][j][xy], s2cur[nb][sj], nzb2cur[nb][sj], q);
    else if constexpr (W8) return dequant_part8<BF16>(wsw[nb][j][xy], wlo[nb][j][xy], scur[nb][sj], zcur[nb][sj], q);
    else if constexpr (HP) return dequant_pair_h(wsw[nb][j][xy], s2cur[nb][sj], nzb2cur[nb][sj], q);
    else return dequant_part<BF16>(wsw[nb][j][xy], scur[nb][sj], zcur[nb][sj], q);
  };

  v16f acc[WMB][WNB];
#pragma unroll
  for (int i = 0; i < WMB; ++i)
#pragma unroll
    for (int nb = 0; nb < WNB; ++nb)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][nb][e] = 0.f;

  // operand reads of slice s4 = 2 jj + xy of a step (jj = word of the step, xy = X' / Y'): row lane & 31 of a 32-row block,
  // 16-byte chunk 4 jj + 2 (lane >> 5) + xy of its 128-byte row
  uint32_t coff[4];
#pragma unroll
  for (int s4 = 0; s4 < 4; ++s4) {
    const int chunk = 4 * (s4 >> 1) + 2 * (lane >> 5) + (s4 & 1);
    coff[s4] = (uint32_t)(kg * (BM * 128) + ((lane & 31) >> 1) * 256 + ((((lane & 1) * 8 + chunk) ^ ((lane >> 1) & 15)) * 16));
  }

  v4u af[DEEP ? 2 : 1][WMB];      // B operands (activations) of the current slice, with DEEP also of the next, refilled in place
  v4u wf[2][WNB];    // A operands (weights) of the current and of the next slice

  // One k-slice: its MFMAs, with the reads of a later slice's activation fragments (slice next_s4 of the step in `next_a`) and the dequantisation of the next
  // one's weights in their shadow.
  auto slice = [&](auto cbuf_c, const uint8_t* next_a, auto next_s4_c, auto next_j_c, auto requests) {
    constexpr int cbuf = decltype(cbuf_c)::value, nbuf = cbuf ^ 1;
    constexpr int next_s4 = decltype(next_s4_c)::value, next_j = decltype(next_j_c)::value, next_xy = (cbuf + 1) & 1, ab = DEEP ? cbuf : 0;
#pragma unroll
    for (int mb = 0; mb < WMB; ++mb) {
#pragma unroll
      for (int nb = 0; nb < WNB; ++nb) acc[mb][nb] = T::mfma32(wf[cbuf][nb], af[ab][mb], acc[mb][nb]);      // rows = n, columns = m
      af[ab][mb] = *reinterpret_cast<const v4u*>(next_a + mb * 4096 + coff[next_s4]);
#pragma unroll
      for (int x = mb * 4 * WNB / WMB; x < (mb + 1) * 4 * WNB / WMB; ++x) wf[nbuf][x >> 2][x & 3] = dequant_q(x >> 2, next_j, next_xy, x & 3);
      if (mb == 0) requests();
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  using C0 = std::integral_constant<int, 0>;
  using C1 = std::integral_constant<int, 1>;
  using C2 = std::integral_constant<int, 2>;
  using C3 = std::integral_constant<int, 3>;

  // Vector-memory operations retire in issue order.  At the barrier of step h, ahead of its last slice (with DEEP of its last two), the activations of step h + 1
  // must have landed; newer than they are those of the NST - 2 steps behind them, the last of whose quarters went out in the slice ahead of it, and the weights requested since.
  constexpr int WAIT = (NST - 2) * A_LD + KW * ((NST - 2) / 2);
  static_assert(NST % 2 == 0 && NST <= 2 * PD, "requests newer than a step's activations: the same for even and odd steps, and in the prologue");
  static_assert(WAIT <= 63 && (NST - 2) * A_LD + (PD - 1) * KW <= 63, "wait counter range");

  // A step's requests (activations of the step NST ahead into the stage that its barrier has freed, on odd steps the weights
  // of the round PD ahead) are spread over the four slices behind the barrier: all at once they fill the memory pipe's queue
  // and every wavefront stalls on it with its matrix instructions behind.
  auto quarter = [&](int h, int stage, int q) { issue_a(h, stage, q * A_LD / 4, (q + 1) * A_LD / 4); };

  // ---- prologue: the requests of the first NST steps (of the last a quarter, with DEEP two: as many as stand behind a barrier in the loop) and PD rounds.  Behind the activations of a step
  // there must be as many requests as in the loop, where round x's weights go out behind step 2 (x - PD) + NST - 2: the waits in
  // front of the barriers count on it. ----
  auto keep_order = [] { asm volatile("" ::: "memory"); __builtin_amdgcn_sched_barrier(0); };
  issue_a(0, 0, 0, A_LD);
  load_w(ring[0], 0);
  keep_order();
#pragma unroll
  for (int h = 1; h < NST - 1; ++h) {
    issue_a(h, h, 0, A_LD);
    keep_order();
#pragma unroll
    for (int x = 1; x < PD; ++x)
      if (h == (x > 2 * (x - PD) + NST - 2 ? x : 2 * (x - PD) + NST - 2)) load_w(ring[x], x);
    keep_order();
  }
#pragma unroll
  for (int x = NST - 1; x < PD; ++x) load_w(ring[x], x);
  keep_order();
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 2) * A_LD + (PD - 1) * KW) : "memory");      // step 0 and the first weights
  advance_w(ring[0]);
  quarter(NST - 1, NST - 1, 0);
  if (DEEP) quarter(NST - 1, NST - 1, 1);
#pragma unroll
  for (int x = 0; x < 4 * WNB; ++x) wf[0][x >> 2][x & 3] = dequant_q(x >> 2, 0, 0, x & 3);
  asm volatile("s_barrier" ::: "memory");
#pragma unroll
  for (int mb = 0; mb < WMB; ++mb) af[0][mb] = *reinterpret_cast<const v4u*>(lds8 + mb * 4096 + coff[0]);
  if constexpr (DEEP) {
#pragma unroll
    for (int mb = 0; mb < WMB; ++mb) af[1][mb] = *reinterpret_cast<const v4u*>(lds8 + mb * 4096 + coff[1]);
  }

  int cur = 0;       // stage of the current step
  auto next_stage = [](int x) { return x + 1 == NST ? 0 : x + 1; };
  auto nothing = [] {};
  // a round: the two steps of this wavefront's group; `fly` = ring slot that is being refilled, `nxt` = the next round's
  // (`last_c`: the rounds behind the loop request no more weights, and count on none -- unused ones the compiler would drop)
  auto round = [&](int r, WSet& fly, WSet& nxt, auto last_c) {
    constexpr bool last = decltype(last_c)::value;
    auto weights = [&](int q) {
      if constexpr (!last) load_w_q(fly, r + PD, q);
    };
    auto step_end = [&] {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(last ? (NST - 2) * A_LD : WAIT) : "memory");
    };
    const uint8_t* A0 = lds8 + cur * STAGE;
    const int s1 = next_stage(cur), s2 = next_stage(s1), sp = cur == 0 ? NST - 1 : cur - 1;
    const uint8_t* A1 = lds8 + s1 * STAGE;
    const uint8_t* A2 = lds8 + s2 * STAGE;
    const int ha = 2 * r - 1 + NST;
    if constexpr (DEEP) {      // (the barrier stands where the next step's first fragments are read, here ahead of the last two slices)
      slice(C0{}, A0, C2{}, C0{}, [&] { weights(0); weights(1); quarter(ha, sp, 2); });
      slice(C1{}, A0, C3{}, C1{}, [&] { weights(2); weights(3); quarter(ha, sp, 3); });
      step_end();
      slice(C0{}, A1, C0{}, C1{}, [&] { quarter(ha + 1, cur, 0); });
      slice(C1{}, A1, C1{}, C2{}, [&] { quarter(ha + 1, cur, 1); });
      slice(C0{}, A1, C2{}, C2{}, [&] { quarter(ha + 1, cur, 2); });
      slice(C1{}, A1, C3{}, C3{}, [&] { quarter(ha + 1, cur, 3); });
      step_end();
      slice(C0{}, A2, C0{}, C3{}, [&] { quarter(ha + 2, s1, 0); });
      advance_w(nxt);
      __builtin_amdgcn_sched_barrier(0);
      slice(C1{}, A2, C1{}, C0{}, [&] { quarter(ha + 2, s1, 1); });
    } else {
      slice(C0{}, A0, C1{}, C0{}, [&] { weights(0); weights(1); quarter(ha, sp, 1); });
      slice(C1{}, A0, C2{}, C1{}, [&] { weights(2); quarter(ha, sp, 2); });
      slice(C0{}, A0, C3{}, C1{}, [&] { weights(3); quarter(ha, sp, 3); });
      step_end();
      slice(C1{}, A1, C0{}, C2{}, [&] { quarter(ha + 1, cur, 0); });
      slice(C0{}, A1, C1{}, C2{}, [&] { quarter(ha + 1, cur, 1); });
      slice(C1{}, A1, C2{}, C3{}, [&] { quarter(ha + 1, cur, 2); });
      slice(C0{}, A1, C3{}, C3{}, [&] { quarter(ha + 1, cur, 3); });
      step_end();
      // the operands of the group's last slice are in wf[1] already: the next words become current in front of it
      advance_w(nxt);
      __builtin_amdgcn_sched_barrier(0);
      slice(C1{}, A2, C0{}, C0{}, [&] { quarter(ha + 2, s1, 0); });
    }
    cur = s2;
  };
  int r = 0;
  static_assert(PD == 2 || PD == 4, "the loop is written out for a ring of two or four");
  // (in multiples of the ring, the rest behind: with exits in the loop's middle the compiler waits for weights of later rounds)
  using IN_LOOP = std::false_type;
  using BEHIND = std::true_type;
  for (; r + PD <= t_full; r += PD) {
    round(r, ring[0], ring[1], IN_LOOP{});
    if constexpr (PD == 2) {
      round(r + 1, ring[1], ring[0], IN_LOOP{});
    } else {
      round(r + 1, ring[1], ring[2], IN_LOOP{});
      round(r + 2, ring[2], ring[3], IN_LOOP{});
      round(r + 3, ring[3], ring[0], IN_LOOP{});
    }
  }
  if (r < t_full) {
    round(r, ring[0], ring[1], BEHIND{});
    if constexpr (PD == 4) {
      if (r + 1 < t_full) {
        round(r + 1, ring[1], ring[2], BEHIND{});
        if (r + 2 < t_full) round(r + 2, ring[2], ring[3], BEHIND{});
      }
    }
  }
  if (rem > 0) {      // the last round, without the wavefronts whose K group lies past the end
    const uint8_t* A0 = lds8 + cur * STAGE;
    const uint8_t* A1 = lds8 + next_stage(cur) * STAGE;
    auto drained = [] { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    auto last_slice = [&](auto cbuf_c) {
      constexpr int cbuf = decltype(cbuf_c)::value;
#pragma unroll
      for (int mb = 0; mb < WMB; ++mb)
#pragma unroll
        for (int nb = 0; nb < WNB; ++nb) acc[mb][nb] = T::mfma32(wf[cbuf][nb], af[DEEP ? cbuf : 0][mb], acc[mb][nb]);
    };
    if (kg < rem) {
      if constexpr (DEEP) {
        slice(C0{}, A0, C2{}, C0{}, nothing);
        slice(C1{}, A0, C3{}, C1{}, nothing);
      } else {
        slice(C0{}, A0, C1{}, C0{}, nothing);
        slice(C1{}, A0, C2{}, C1{}, nothing);
        slice(C0{}, A0, C3{}, C1{}, nothing);
      }
    }
    drained();
    if (kg < rem) {
      if constexpr (DEEP) {
        slice(C0{}, A1, C0{}, C1{}, nothing);
        slice(C1{}, A1, C1{}, C2{}, nothing);
        slice(C0{}, A1, C2{}, C2{}, nothing);
        slice(C1{}, A1, C3{}, C3{}, nothing);
        slice(C0{}, A1, C3{}, C3{}, nothing);      // (reads a slice again that nobody uses)
      } else {
        slice(C1{}, A1, C0{}, C2{}, nothing);
        slice(C0{}, A1, C1{}, C2{}, nothing);
        slice(C1{}, A1, C2{}, C3{}, nothing);
        slice(C0{}, A1, C3{}, C3{}, nothing);
      }
      last_slice(C1{});
    }
  }
  // every wavefront is done with the stages and nothing is on its way into them: the partial sums may use the LDS
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

  // ---- the KG partial sums of a strip: a wavefront adds up 1 / KG of its strip's 16-byte pieces, in the order of the K groups ----
  constexpr int PIECES = WMB * WNB * 4, OWN = PIECES / KG;      // piece = 4 * (WNB * m-block + column block) + quarter (8 columns)
  v4f sum[OWN];
  auto piece = [&](int c) { return v4f{acc[c / (4 * WNB)][c / 4 % WNB][4 * (c % 4)], acc[c / (4 * WNB)][c / 4 % WNB][4 * (c % 4) + 1],
                                       acc[c / (4 * WNB)][c / 4 % WNB][4 * (c % 4) + 2], acc[c / (4 * WNB)][c / 4 % WNB][4 * (c % 4) + 3]}; };
  // slot of K group `from`'s contribution to K group `to`'s pieces
  auto slot = [&](int to, int from) { return lds8 + (((to * (KG - 1) + from - (from > to)) * NS + ns) * OWN) * 1024 + lane * 16; };
#pragma unroll
  for (int k = 0; k < KG; ++k) {
    if (k == kg) {
#pragma unroll
      for (int c = 0; c < OWN; ++c) sum[c] = piece(k * OWN + c);
    } else {
      uint8_t* d = slot(k, kg);
#pragma unroll
      for (int c = 0; c < OWN; ++c) *reinterpret_cast<v4f*>(d + c * 1024) = piece(k * OWN + c);
    }
  }
  if constexpr (KG > 1) {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if constexpr (KG == 2) {      // (the sum of two does not depend on their order)
#pragma unroll
      for (int c = 0; c < OWN; ++c) sum[c] += *reinterpret_cast<const v4f*>(slot(kg, 1 - kg) + c * 1024);
    } else {
#pragma unroll
      for (int c = 0; c < OWN; ++c) {
        v4f total = v4f{0.f, 0.f, 0.f, 0.f};
        for (int k = 0; k < KG; ++k) total += k == kg ? sum[c] : *reinterpret_cast<const v4f*>(slot(kg, k == kg ? (kg + 1) % KG : k) + c * 1024);
        sum[c] = total;
      }
    }
  }
  const int own0 = kg * OWN;
  if (sl.nsplit > 1 && !handover_pieces<OWN, NW>(p.c_tmp, p.counters, sum, sl, wave, lane)) return;

  // ---- bias, rounding, stores: a piece holds 8 columns of row lane & 31 of its block, columns 4 * (lane >> 5) + 0..3 of them in
  // this lane; two pieces exchange their halves across the lanes so that every lane stores 16 bytes of one row ----
  const int nb0 = n0 + ns * TN;
  constexpr int PAIR = OWN % 2 ? 1 : 2;
  const bool wide = PAIR == 2 && ((uintptr_t)p.c & 15) == 0;
#pragma unroll
  for (int c = 0; c < OWN; c += PAIR) {
    v2u pk[PAIR];
    const int pc = own0 + c, mrow = m0 + 32 * (pc / (4 * WNB)) + (lane & 31), nc = nb0 + 32 * (pc / 4 % WNB) + 8 * (pc & 3);
    if (nc >= p.N) continue;
#pragma unroll
    for (int x = 0; x < PAIR; ++x) {
      v4f v = sum[c + x];
      if (p.bias) {
        const v2u bb = *reinterpret_cast<const v2u*>(p.bias + nc + 8 * x + 4 * (lane >> 5));
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
      const auto s0 = __builtin_amdgcn_permlane32_swap(pk[0].x, pk[PAIR - 1].x, false, false);
      const auto s1 = __builtin_amdgcn_permlane32_swap(pk[0].y, pk[PAIR - 1].y, false, false);
      if (mrow < p.M) *reinterpret_cast<v4u*>(row + 8 * (lane >> 5)) = v4u{s0[0], s1[0], s0[1], s1[1]};
    } else {
#pragma unroll
      for (int x = 0; x < PAIR; ++x) *reinterpret_cast<v2u*>(row + 8 * x + 4 * (lane >> 5)) = pk[x];
    }
  }
}

template <bool BF16, int WMB, int WNB, int NS, bool HAS_ZP, int SUBG, bool W8, int NST, int PD>
static int launch_strip(const PrefillParams& p_in, hipStream_t s) {
  PrefillParams p = p_in;
  constexpr size_t lds = strip_lds_bytes<WMB, WNB, NS>(NST);
  static_assert(lds <= 160 * 1024, "LDS");
  auto kern = w4a16_strip_kernel<BF16, WMB, WNB, NS, HAS_ZP, SUBG, W8, NST, PD>;
  static size_t reserved[VAQ_MAX_DEVICES];
  if (const int rc = reserve_dynamic_lds(reinterpret_cast<const void*>(kern), lds, reserved, "w4a16_gemm(strip)"); rc != VAQ_OK) return rc;
  const int tiles_m = (p.M + 32 * WMB - 1) / (32 * WMB), tiles_n = (p.N + 32 * WNB * NS - 1) / (32 * WNB * NS), tiles = tiles_m * tiles_n;
  const KernelHead h = prefill_head(p, tile_grid(tiles_m, tiles_n, p.SK, p.tail_first));
  p.split_magic = tile_split_magic(tiles, p.SK, p.tail_first);
  const dim3 grid = p.tail_first > 0 ? dim3(p.tail_first + (tiles - p.tail_first) * p.SK) : dim3(tiles, p.SK);
  hipLaunchKernelGGL(kern, grid, dim3(512), lds, s, h.a, h.b, h.c, p);
  return VAQ_OK;
}

// The shapes, by tile id; which one a problem takes is priced (w4a16_prefill.hip).  64 .. 128 KiB of stages; a ring of two where four
// do not fit the registers.
template <bool BF16, bool HAS_ZP, int SUBG, bool W8>
static int strip_dispatch(const PrefillParams& p, int tile, hipStream_t s) {
  constexpr bool WIDE = SUBG == 1 && !W8;      // (the widest shapes need the registers that sub-groups and second blocks take)
  switch (tile) {
    case 41: return launch_strip<BF16, 1, 1, 4, HAS_ZP, SUBG, W8, 8, 4>(p, s);      //  32 x 128
    case 42: return launch_strip<BF16, 2, 1, 4, HAS_ZP, SUBG, W8, 4, 4>(p, s);      //  64 x 128
    case 43: return launch_strip<BF16, 3, 1, 4, HAS_ZP, SUBG, W8, 4, SUBG == 4 ? 2 : 4>(p, s);      //  96 x 128
    case 44: return launch_strip<BF16, 4, 1, 4, HAS_ZP, SUBG, W8, 4, WIDE ? 4 : 2>(p, s);      // 128 x 128
    case 46: return launch_strip<BF16, 4, 1, 8, HAS_ZP, SUBG, W8, 4, WIDE ? 4 : 2>(p, s);      // 128 x 256, eight strips of 32 columns
    case 51: return launch_strip<BF16, 1, 1, 2, HAS_ZP, SUBG, W8, 4, SUBG == 4 ? 2 : 4>(p, s);      //  32 x 64
    case 52: return launch_strip<BF16, 2, 1, 2, HAS_ZP, SUBG, W8, 4, WIDE ? 4 : 2>(p, s);      //  64 x 64
    case 66:
      if constexpr (WIDE) return launch_strip<BF16, 4, 2, 4, HAS_ZP, SUBG, W8, 4, 2>(p, s);      // 128 x 256
      break;
    default: break;
  }
  set_error("w4a16_gemm(strip): tile id %d is not built for this weight format", tile);
  return VAQ_ERR_UNSUPPORTED;
}

}  // namespace vaq
