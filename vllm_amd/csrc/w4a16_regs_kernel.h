// W4A16 GEMM for a few to some dozen rows, weights and activations in registers: C[M,N] = A[M,K] . dequant(B[K,N]) (+bias), the
// arithmetic of w4a16_decode.hip (codes as exact 16-bit numbers BIAS + code, 8-bit ones in bf16 without bias; zero point and group scale in fp32 on the accumulator).
//
//  * A wavefront multiplies one k-tile (128 rows of K) of its rows with J neighbouring n-tiles at a time.  What the kernel that stages a
//    slab of activations once per workgroup (w4a16_decode2_kernel.h) pays from 17 rows on -- one LDS operand read per MFMA (6 us of the
//    21 us that 4096 x 28672 takes at M = 32), and a hand-over between workgroups where the slab does not fit LDS -- falls by J: the
//    operands of a k-tile leave LDS once for J tiles, and a wavefront keeps no more of them there than the k-tile to come.
//  * The NW wavefronts of a workgroup take the k-tiles of its part of K in turn and share nothing until their sums meet in LDS at the end:
//    no barrier in the K loop.  Activations, scales and zero points come by direct-to-LDS loads into a piece of LDS of the wavefront's own,
//    weights into a ring of two k-tiles of registers.
//  * The scales of a k-tile are one row of J * 16 columns: one load for all J tiles, requested with the activations.  (One 8-byte load per
//    tile, as the other decode kernels do it, cost 3 us on 4096 x 28672 at M = 16: 32-byte pieces of rows 57 KB apart, and the weights
//    behind them in the queue wait for each: 11.6 us for the weights alone, 14.9 with them.)
//  * Rows beyond MB * 16 are a second block of rows with workgroups of their own, side by side on the same XCD, so that they find the
//    weights in its L2.  K may be split over workgroups: partial tiles and one arrival counter per 16 x 16 result, summed in split order.
//  * Codes with their bias and the correction that takes it out again both overflow where an activation is infinite or close to the largest bf16
//    number: results that are not finite are computed again with the weights themselves (regs_rounded_tile).
//
// Cold, us, the kernel that took them before and this one: 4096 x 28672 at M = 24 / 32 / 48 20.2 / 21.2 / 29.0 -> 17.1 / 16.9 / 21.8;
// 14336 x 4096 at M = 48 / 64 21.7 / 25.7 -> 17.2 / 17.7; 4096 x 6144 at M = 48 / 64 10.1 / 11.0 -> 9.2 / 9.6.
// Not kept: operands straight from memory into registers (pieces of 64 bytes per row: 4096 x 28672 at M = 32 18.5, 14336 x 4096 16.0 us),
// deeper rings (three and four k-tiles: level or slower), a start of the K loop that differs from workgroup to workgroup (+0.3 us), results
// gathered in LDS and stored in whole rows of the range instead of 32-byte pieces (level: one more barrier).
#pragma once
#include "vaq_common.h"

#include <type_traits>

namespace vaq {

struct RegsParams {
  const uint16_t* a;
  const v4u* b;
  const uint16_t* scales;
  const uint32_t* zeros;
  const uint16_t* bias;
  uint16_t* c;
  float* c_tmp;
  int32_t* counters;
  int M, N, lda;
  int G, NT;               // k-tiles of 128 rows, n-tiles of 16 columns
  int SK, RB;              // parts of K, blocks of MB * 16 rows
  int ranges, per_xcd;     // ranges of J n-tiles; workgroups of an XCD
  int s_stride, z_stride;  // elements between consecutive rows of scales (N) / zeros (N/8); 0 for channelwise
  uint32_t k_mask, k_ex;   // 0x000f000f and the exponent pattern, as run-time values (see w4a16_decode.hip)
};

// Counts: rows (up to 256), parts of K (8) and blocks of rows (16) in 9, 4 and 5 bits, and above them 2^12 / blocks, rounded up: x / blocks = x * that >> 12
// for x < 128, a copy's number.  And x / copies = mul_high(x, 2^32 / copies + 1) for the x here, below 2^25.
inline KernelHead regs_head(const RegsParams& p) {
  const uint32_t counts = (uint32_t)p.M | (uint32_t)p.SK << 9 | (uint32_t)p.RB << 13 | (uint32_t)((4096 + p.RB - 1) / p.RB) << 18;
  return KernelHead{v8u{ptr_lo(p.a), ptr_hi(p.a), ptr_lo(p.b), ptr_hi(p.b), ptr_lo(p.scales), ptr_hi(p.scales), (uint32_t)p.lda, (uint32_t)p.G},
                    v4u{(uint32_t)p.NT, counts, (uint32_t)p.ranges, (uint32_t)p.per_xcd},
                    v2u{(uint32_t)p.s_stride, (uint32_t)((1ull << 32) / (uint32_t)(p.SK * p.RB) + 1)}};
}

// What a workgroup computes: one contiguous range of units per XCD; the K parts and row blocks of one range of n-tiles are neighbours.  (No division where K is
// whole: a 32-bit one is some 30 instructions, a 64-bit one more than 100.)  Callable on the host for its test.
struct RegsUnit {
  uint32_t range, sk, rb, g_lo, g_hi;      // range of n-tiles, part of K and its k-tiles, block of rows
};
__host__ __device__ inline uint32_t regs_place(uint32_t block, uint32_t per_xcd) { return (block & 7u) * per_xcd + (block >> 3); }
__host__ __device__ inline RegsUnit regs_unit(uint32_t unit, uint32_t counts, uint32_t copies_magic, uint32_t G) {
  const int SK = (int)(counts >> 9 & 0xfu), RB = (int)(counts >> 13 & 0x1fu);
  const uint32_t copies = (uint32_t)(SK * RB);
  RegsUnit u{unit, 0, 0, 0, G};
  if (copies > 1) {
    u.range = mul_high(unit, copies_magic);
    u.rb = unit - u.range * copies;
    if (SK > 1) {
      u.sk = u.rb * (counts >> 18) >> 12;
      u.rb -= u.sk * (uint32_t)RB;
      u.g_lo = G * u.sk / (uint32_t)SK;
      u.g_hi = G * (u.sk + 1) / (uint32_t)SK;
    }
  }
  return u;
}

constexpr size_t regs_lds_bytes(int mb, int mr, int j, int nw, int sub, bool zp) {
  const size_t run = (size_t)nw * (mb * mr * 256 + 2 * (sub * 256 + (zp ? 256 : 0)));      // activations of a k-tile, scales and zero points of two
  const size_t sums = (size_t)j * mb * nw * 1024;                                      // partial results
  return run > sums ? run : sums;
}

// One 16 x 16 result, all of K, its weights rounded to 16 bits ahead of the product as the tile kernels do it: what a call gets where codes with
// their bias give no finite number.  (inf - inf where the weights' own signs would decide; and of bf16
// activations beyond 2^120 the biased sums overflow, those of the weights do not.)  By one wavefront, without any prefetch:
// 4096 x 28672 at M = 32 takes 144 us with one such row and 18 without.
template <bool BF16, bool HAS_ZP, int SUBG, bool W8>
__device__ __attribute__((always_inline)) inline v4f regs_rounded_tile(const __attribute__((address_space(4))) RegsParams& p, int nt, int row, int lane) {
  using T = F16Traits<BF16>;
  constexpr int PL = W8 ? 2 : 1;
  const int o = lane >> 4, r16 = lane & 15, n = nt * 16 + r16;
  const v4u* const a = reinterpret_cast<const v4u*>(p.a + (int64_t)min(row + r16, p.M - 1) * p.lda) + o;
  v4f sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int g = 0; g < p.G; ++g) {
    const v4u* const word = p.b + (uint32_t)(nt * p.G + g) * (uint32_t)(PL * 64);
    const v4u w = word[(uint32_t)lane], wl = W8 ? word[(uint32_t)lane + 64] : v4u{0u, 0u, 0u, 0u};
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      __builtin_amdgcn_sched_barrier(0);      // (one word after the other: this path is not to set the kernel's register count)
      const v4u act = a[g * 16 + jj * 4];
      const uint32_t q = (uint32_t)(g * SUBG + jj * SUBG / 4);      // (offsets below 2 GiB, as in the K loop)
      const float s = T::to_float((p.scales + q * (uint32_t)p.s_stride)[(uint32_t)n]);
      const int z = HAS_ZP ? (int)((p.zeros + q * (uint32_t)p.z_stride)[(uint32_t)n / 8] >> ((n & 7) * 4) & 0xFu) : W8 ? 128 : 8;
      uint32_t aop[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        auto weight = [&](int at) {
          const uint32_t c = W8 ? (w[jj] >> at & 0xFu) * 16u + (wl[jj] >> at & 0xFu) : w[jj] >> at & 0xFu;
          return (uint32_t)T::from_float((float)((int)c - z) * s);
        };
        aop[i] = weight(4 * i) | weight(4 * i + 16) << 16;
      }
      sum = T::mfma16(v4u{aop[0], aop[1], aop[2], aop[3]}, act, sum);
    }
  }
  return sum;
}

// 8-bit codes of two nibble planes as one operand: 8 codes of consecutive k, in fp16 as 1024 + code (a byte behind the exponent), in bf16, whose 8 bits hold them whole, as they are.
// As two operands, a plane each with its bias and the high one's products times 16, a code took two products, 14 instructions for 8 codes where these are 8 / 16, and four fused ones
// for each result and group where there is one now (in groups of 128 rows; two in smaller ones).  Cold, us: 3584 x 4608 at M = 51 / 64 11.5 / 11.8 -> 10.0 / 10.4, 2048 x 23808 at
// M = 19 in groups of 32 20.2 -> 16.1, 3072 x 16128 at M = 1 12.1 -> 11.5; 300 drawn calls of 1 .. 256 rows 0.963 in the mean, fp16 0.95, bf16 0.97.  Against 64 bits the error
// is level in bf16 and smaller in fp16 (activations around 3 in groups of 128 rows 2.5e-4 -> 2.1e-4: 1024 + code instead of 16 (1024 + high) + 1024 + low).
template <bool BF16>
__device__ inline v4u regs_codes8(uint32_t hi, uint32_t lo) {
  // bytes 0 .. 3: elements 0,4,1,5 and 2,6,3,7
  const uint32_t t = ((hi << 4) & 0xf0f0f0f0u) | (lo & 0x0f0f0f0fu), u = (hi & 0xf0f0f0f0u) | ((lo >> 4) & 0x0f0f0f0fu);
  if constexpr (BF16) {      // (no inline assembly: the compiler keeps clear of a product under way whose unused results share the registers only with its own instructions)
    auto pair = [](uint32_t lo, uint32_t hi) {
      typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
      return __builtin_bit_cast(uint32_t, v2bf{(__bf16)(float)(lo & 0xffu), (__bf16)(float)(hi & 0xffu)});
    };
    return v4u{pair(t, t >> 16), pair(u, u >> 16), pair(t >> 8, t >> 24), pair(u >> 8, u >> 24)};
  }
  return v4u{(t & 0x00ff00ffu) | 0x64006400u, (u & 0x00ff00ffu) | 0x64006400u, __builtin_amdgcn_perm(0x64646464u, t, 0x04030401u),
             __builtin_amdgcn_perm(0x64646464u, u, 0x04030401u)};
}

// The sum of the wavefronts' parts of result q in LDS, and of the parts of K in c_tmp (four in flight, added in split order).
template <int NW>
__device__ __attribute__((always_inline)) inline v4f regs_sum(const v4f* red, int results, int q, int lane) {
  v4f val = red[q * 64 + lane];
#pragma unroll
  for (int s = 1; s < NW; ++s) val += red[(s * results + q) * 64 + lane];
  return val;
}
__device__ __attribute__((always_inline)) inline v4f regs_sum_parts(const __amdgpu_buffer_rsrc_t rt, uint32_t units, uint32_t u, int SK, int lane) {
  v4f val = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < SK; s0 += 4) {
    v4u part[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      part[i] = __builtin_amdgcn_raw_buffer_load_b128(rt, lane * 16, (int)(((uint32_t)min(s0 + i, SK - 1) * units + u) * 1024u), 16);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (s0 + i < SK) val += __builtin_bit_cast(v4f, part[i]);
  }
  return val;
}
template <bool BF16, class Params>
__device__ __attribute__((always_inline)) inline void regs_store(const Params& p, v4f val, int m, int n) {
  using T = F16Traits<BF16>;
  if (p.bias) {
    const v2u bb = *reinterpret_cast<const v2u*>(p.bias + n);
    val[0] += T::to_float((uint16_t)(bb.x & 0xffffu));
    val[1] += T::to_float((uint16_t)(bb.x >> 16));
    val[2] += T::to_float((uint16_t)(bb.y & 0xffffu));
    val[3] += T::to_float((uint16_t)(bb.y >> 16));
  }
  v2u outv;
  outv.x = (uint32_t)T::from_float(val[0]) | ((uint32_t)T::from_float(val[1]) << 16);
  outv.y = (uint32_t)T::from_float(val[2]) | ((uint32_t)T::from_float(val[3]) << 16);
  if (m < p.M) *reinterpret_cast<v2u*>(p.c + (int64_t)m * p.N + n) = outv;
}

// MR: rows of an m-block that are fetched, 16 or, of a single one, 4 (columns of the MFMAs are independent: those of the other rows read a
// row that is there, and their results are not stored).  SUBG: quantisation groups per k-tile (1, 2, 4).  W8: 8-bit codes, two nibble planes in memory.  OCC: wavefronts per SIMD that the registers
// are to allow.
template <bool BF16, int MB, int MR, int J, bool HAS_ZP, int NW, int SUBG, bool W8, int OCC>
__global__ __launch_bounds__(NW * 64, OCC) void w4a16_regs_kernel(VAQ_HEAD_ARGS, const RegsParams p) {
  // what the first requests need (see regs_head)
  const uint16_t* const a = head_ptr<uint16_t>(h0[0], h0[1]);
  const v4u* const b = head_ptr<v4u>(h0[2], h0[3]);
  const uint16_t* const scales = head_ptr<uint16_t>(h0[4], h0[5]);
  const uint32_t lda = h0[6], G = h0[7], NT = h1[0], counts = h1[1], ranges = h1[2], per_xcd = h1[3], s_stride = h2[0], copies_magic = h2[1];
  using T = F16Traits<BF16>;
  static_assert(!(W8 && HAS_ZP), "8-bit codes have no zero points");
  static_assert(MR == 16 || (MR == 4 && MB == 1), "fewer rows of a single m-block only");
  constexpr int PL = W8 ? 2 : 1;      // planes of codes
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int o = lane >> 4, r16 = lane & 15;
  const int M = (int)(counts & 0x1ffu), SK = (int)(counts >> 9 & 0xfu), RB = (int)(counts >> 13 & 0x1fu);
  const uint32_t unit = regs_place(blockIdx.x, per_xcd);
  if (unit >= ranges * (uint32_t)(SK * RB)) return;
  const RegsUnit u = regs_unit(unit, counts, copies_magic, G);
  const uint32_t range = u.range, sk = u.sk;
  const int rb_i = (int)u.rb, g_lo = (int)u.g_lo, g_hi = (int)u.g_hi;
  const int nt0 = (int)range * J, row0 = rb_i * MB * 16;

  auto rsrc = [](const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
  };
  // (the extents are those of RegsParams)
  const __amdgpu_buffer_rsrc_t ra = rsrc(a, ((uint32_t)(M - 1) * lda + G * 128u) * 2u), rb = rsrc(b, NT * G * (uint32_t)(PL * 1024));
  const uint32_t s_bytes = (s_stride ? G * (uint32_t)SUBG : 1u) * NT * 32u;
  const __amdgpu_buffer_rsrc_t rs = rsrc(scales, s_bytes), rz = HAS_ZP ? rsrc(p.zeros, s_bytes / 4) : rs;

  // This wavefront's piece of LDS: the activations of the next k-tile, MR * MB rows of 256 bytes with chunk c of row r at place
  // c ^ (r & 15); scales (256 bytes per group row) and zero points (64 per row, one piece) of the k-tile at hand and the next.
  constexpr int AI = MB * MR / 4, ACT = AI * 1024, SC = SUBG * 256, SIDE = SC + (HAS_ZP ? 256 : 0), OWN = ACT + 2 * SIDE;
  uint8_t* const mine = lds + (size_t)w * OWN;
  uint32_t vo_a[AI];      // instruction i fetches rows 4i .. 4i + 3
#pragma unroll
  for (int i = 0; i < AI; ++i) {
    const int r = i * 4 + o;
    vo_a[i] = (uint32_t)min(row0 + r, M - 1) * lda * 2u + (uint32_t)((r16 ^ (r & 15)) * 16);
  }
  constexpr uint32_t OUT = 0x80000000u;      // past the end of every buffer: reads as zero
  struct At {                                // a k-tile: its number, or 0 and OUT for none
    uint32_t g, out;
  };
  auto at = [&](int g) { return At{g < g_hi ? (uint32_t)g : 0u, g < g_hi ? 0u : OUT}; };
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  auto load_act = [&](int s, At t) {      // for slot s of the ring
#pragma unroll
    for (int i = 0; i < AI; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(mine + i * 1024), 16, (int)(vo_a[i] | t.out), (int)(t.g * 256u), 0, 0);
    uint8_t* const side = mine + ACT + s * SIDE;
#pragma unroll
    for (int sj = 0; sj < SUBG; ++sj)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(side + sj * 256), 4, (int)((lane < J * 8 ? (uint32_t)lane * 4u : OUT) | t.out),
                                               (int)(((t.g * SUBG + sj) * s_stride + (uint32_t)nt0 * 16u) * 2u), 0, 0);
    if constexpr (HAS_ZP) {      // 16 lanes a row
      const uint32_t vo = o < SUBG && r16 < J * 2 ? (uint32_t)o * (uint32_t)p.z_stride * 4u + (uint32_t)r16 * 4u : OUT;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rz, (lds_ptr_t)(side + SC), 4, (int)(vo | t.out),
                                               (int)((t.g * SUBG * (uint32_t)p.z_stride + (uint32_t)nt0 * 2u) * 4u), 0, 0);
    }
  };
  v4u wq[2][J][PL];
  auto load_w = [&](int s, At t, int j) {
    const uint32_t nt = (uint32_t)min(nt0 + j, (int)NT - 1);
#pragma unroll
    for (int pl = 0; pl < PL; ++pl)
      wq[s][j][pl] = __builtin_amdgcn_raw_buffer_load_b128(rb, (int)((uint32_t)lane * 16u | t.out), (int)(((nt * G + t.g) * PL + pl) * 1024u), 2);
  };

  v4f acc[J][MB];
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[j][mb] = v4f{0.f, 0.f, 0.f, 0.f};

  uint32_t ex;
  asm volatile("v_mov_b32 %0, %1" : "=v"(ex) : "s"(p.k_ex));
  const uint32_t msk = p.k_mask;

  // The k-tile in slot s.  Behind it are requested, as soon as there is room: the next one's activations, then tile by tile the weights of
  // the one after that (the scheduling barriers keep each weight request behind the arithmetic that frees its registers, which is what
  // saves copying them).
  auto tile = [&](int s, bool refill_act, At next_act, bool refill_w, At next_w) {
    v4u act[4][MB];
    const uint8_t* const side = mine + ACT + s * SIDE;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj)
        act[jj][mb] = *reinterpret_cast<const v4u*>(mine + mb * 4096 + (r16 & (MR - 1)) * 256 + (((jj * 4 + o) ^ (r16 & (MR - 1))) * 16));
    if (refill_act) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // this tile's are in registers
      __builtin_amdgcn_sched_barrier(0);
      load_act(s ^ 1, next_act);
      __builtin_amdgcn_sched_barrier(0);
    }
    // row sums S of each group: the same in the four registers.  What every code has too much (regs_codes8) times S is taken out where the group's chain of products starts, zero
    // points of the groups' own behind it, together with the bias where the registers hold no starts (NO_START).  (As a fused operation for every result, n-tile and group 248 drawn
    // calls in groups of 64 / 32 rows without zero points take 1.02 of the time; bias and zero points in one, converted nibble by nibble, 270 with zero points 1.013, in groups of 32 1.03.)
    constexpr bool NO_START = HAS_ZP && SUBG > 1 && (MB == 3 || MB * J >= 16);
    constexpr float ZERO = W8 ? (BF16 ? 128.0f : T::CODE_BIAS + 128.0f) : HAS_ZP ? T::CODE_BIAS : T::CODE_BIAS + 8.0f;
    v4f start[NO_START ? 1 : SUBG][MB];
    float S[SUBG][MB];
    const v4u ones = {T::ONE2, T::ONE2, T::ONE2, T::ONE2};
#pragma unroll
    for (int sj = 0; sj < SUBG; ++sj)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        v4f t = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int jj = sj * (4 / SUBG); jj < (sj + 1) * (4 / SUBG); ++jj) t = T::mfma16(ones, act[jj][mb], t);
        if constexpr (!NO_START) start[sj][mb] = t * -ZERO;
        S[sj][mb] = t[0];
      }
#pragma unroll
    for (int j = 0; j < J; ++j) {
#pragma unroll
      for (int sj = 0; sj < SUBG; ++sj) {
        const v2u sct = *reinterpret_cast<const v2u*>(side + sj * 256 + j * 32 + o * 8);
        const uint32_t z4 = HAS_ZP ? *reinterpret_cast<const uint32_t*>(side + SC + sj * 64 + j * 8 + (o >> 1) * 4) >> ((o & 1) * 16) : 0u;
        v4f P[MB];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) P[mb] = NO_START ? v4f{0.f, 0.f, 0.f, 0.f} : start[NO_START ? 0 : sj][mb];
#pragma unroll
        for (int jj = sj * (4 / SUBG); jj < (sj + 1) * (4 / SUBG); ++jj) {
          const uint32_t wj = wq[s][j][0][jj];
          v4u aop;
          if constexpr (W8) {
            aop = regs_codes8<BF16>(wj, wq[s][j][PL - 1][jj]);
          } else {
            aop.x = (wj & msk) | ex;
            aop.y = ((wj >> 4) & msk) | ex;
            aop.z = ((wj >> 8) & msk) | ex;
            aop.w = ((wj >> 12) & msk) | ex;
          }
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) P[mb] = T::mfma16(aop, act[jj][mb], P[mb]);
        }
        float sf[4];
        if constexpr (BF16) {
          sf[0] = __uint_as_float(sct.x << 16);
          sf[1] = __uint_as_float(sct.x & 0xffff0000u);
          sf[2] = __uint_as_float(sct.y << 16);
          sf[3] = __uint_as_float(sct.y & 0xffff0000u);
        } else {
          sf[0] = T::to_float((uint16_t)(sct.x & 0xffffu));
          sf[1] = T::to_float((uint16_t)(sct.x >> 16));
          sf[2] = T::to_float((uint16_t)(sct.y & 0xffffu));
          sf[3] = T::to_float((uint16_t)(sct.y >> 16));
        }
        float zf[4] = {0.f, 0.f, 0.f, 0.f};
        if constexpr (HAS_ZP) {
          const uint32_t even = z4 & 0x0f0fu, odd = z4 >> 4 & 0x0f0fu;
          zf[0] = (float)(even & 0xffu);
          zf[1] = (float)(odd & 0xffu);
          zf[2] = (float)(even >> 8);
          zf[3] = (float)(odd >> 8 & 0xffu);
        }
        if constexpr (NO_START) {
#pragma unroll
          for (int r = 0; r < 4; ++r) zf[r] += ZERO;
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) acc[j][mb][r] = fmaf(sf[r], HAS_ZP ? fmaf(-zf[r], S[sj][mb], P[mb][r]) : P[mb][r], acc[j][mb][r]);
        }
      }
      if (refill_w) {
        __builtin_amdgcn_sched_barrier(0);
        load_w(s, next_w, j);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  // This wavefront's k-tiles: g_lo + w + i * NW.  The order of the requests is W(0) A(0) W(1) | A(1) W(2) | A(2) W(3) | ..., `|` = a tile:
  // a tile starts when all but the weights requested behind its activations have been answered.
  auto wait = [&] { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(J * PL) : "memory"); };
  int g = g_lo + w;
#pragma unroll
  for (int j = 0; j < J; ++j) load_w(0, at(g), j);
  __builtin_amdgcn_sched_barrier(0);
  load_act(0, at(g));
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int j = 0; j < J; ++j) load_w(1, at(g + NW), j);
  __builtin_amdgcn_sched_barrier(0);
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("" ::"s"(msk), "s"(p.bias), "s"(p.c), "s"(p.c_tmp), "s"(p.counters), "s"(p.N), "s"(p.NT));      // (arrived before the K loop: with
  // a scalar load under way its waits for LDS reads are for all of them at once, and loads ahead of the last k-tile were waited for; 0.1 us)
#endif
#pragma unroll 1
  for (; g + NW < g_hi; g += 2 * NW) {
    wait();
    tile(0, true, at(g + NW), true, at(g + 2 * NW));
    wait();
    tile(1, true, at(g + 2 * NW), true, at(g + 3 * NW));
  }
  if (g < g_hi) {
    wait();
    tile(0, false, At{0u, OUT}, false, At{0u, OUT});
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // (what is requested past the end writes zeros into LDS)

  // ---- the wavefronts' parts of K, on top of the activations ----
  const int here = (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));      // the lane, not kept over the K loop
  v4f* const red = reinterpret_cast<v4f*>(lds);                                       // [NW][J * MB][64]
  __syncthreads();
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) red[(w * (J * MB) + j * MB + mb) * 64 + here] = acc[j][mb];
  __syncthreads();
  uint32_t odd = 0;      // a bit for each result of this wavefront that is not finite
  for (int q = w, bit = 1; q < J * MB; q += NW, bit <<= 1) {
    const int j = q / MB, mb = q - j * MB;
    const int nt = nt0 + j;
    if (nt >= p.NT || row0 + mb * 16 >= p.M) continue;
    v4f val = regs_sum<NW>(red, J * MB, q, here);
    if (SK > 1) {
      // partial tiles and counters as in w4a16_decode2_kernel.h, step 5
      const uint32_t units = (uint32_t)p.NT * (uint32_t)(p.RB * MB), u = (uint32_t)nt * (uint32_t)(p.RB * MB) + (uint32_t)(rb_i * MB + mb);
      const __amdgpu_buffer_rsrc_t rt = rsrc(p.c_tmp, units * 1024u * (uint32_t)p.SK);
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, val), rt, here * 16, (int)(((uint32_t)sk * units + u) * 1024u), 16);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // partial tile acknowledged before the counter moves
      int old = 0;
      if (here == 0) old = __hip_atomic_fetch_add(&p.counters[u], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      old = __builtin_amdgcn_readfirstlane(old);
      if (old != p.SK - 1) continue;
      val = regs_sum_parts(rt, units, u, p.SK, here);
      if (here == 0) __hip_atomic_store(&p.counters[u], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    regs_store<BF16>(p, val, row0 + mb * 16 + (here & 15), nt * 16 + (here >> 4) * 4);
    const float all = fabsf(val[0]) + fabsf(val[1]) + fabsf(val[2]) + fabsf(val[3]);
    odd |= __ballot(!__builtin_isfinite(all)) != 0 ? (uint32_t)bit : 0u;
  }
  if (__builtin_expect(odd != 0, 0)) {
    // The results that are not finite once more, behind their stores.  The arguments are read again and everything is made from values that a statement
    // hides, so that nothing of this is computed, or kept in registers, ahead.  (Tested ahead of each store,
    // or with the path inside the loop over results, calls that go to this kernel took 1.002 .. 1.006 of their time in the mean; in a function that is called 1.006; so
    // 0.997.)  The pointer is the kernel's; in a function that is called it
    // would be null.
    auto args = __builtin_amdgcn_kernarg_segment_ptr();
    int q = w, nt_h = nt0, row_h = row0, rb_h = rb_i;
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("" : "+s"(args), "+s"(q), "+s"(nt_h), "+s"(row_h), "+s"(rb_h));
#endif
    const auto& pa = *(const __attribute__((address_space(4))) RegsParams*)((const __attribute__((address_space(4))) char*)args + HEAD_BYTES);
#pragma unroll 1
    for (; odd != 0; q += NW, odd >>= 1) {
      if (!(odd & 1u)) continue;
      const int j = q / MB, mb = q - j * MB, nt = nt_h + j, row = row_h + mb * 16;
      const uint32_t units = (uint32_t)pa.NT * (uint32_t)(pa.RB * MB), u = (uint32_t)nt * (uint32_t)(pa.RB * MB) + (uint32_t)(rb_h * MB + mb);
      v4f val = pa.SK > 1 ? regs_sum_parts(rsrc(pa.c_tmp, units * 1024u * (uint32_t)pa.SK), units, u, pa.SK, here) : regs_sum<NW>(red, J * MB, q, here);
      const v4f again = regs_rounded_tile<BF16, HAS_ZP, SUBG, W8>(pa, nt, row, here);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (!__builtin_isfinite(val[r])) val[r] = again[r];
      regs_store<BF16>(pa, val, row + (here & 15), nt * 16 + (here >> 4) * 4);
    }
  }
}

// Registers of a lane as the prices count them (they are fitted on it): two k-tiles of weights, sums, operands, a chain per plane, row sums.  8-bit codes have one chain now and, like groups of 64 / 32 rows
// of 4-bit codes, starts of their own: against the compiled instances this is up to 39 too many for 8-bit codes, 21 too few to 38 too many for 4-bit ones; counted as compiled, with another fit or without,
// the plans are no better.  Above 256 sums lie in accumulation registers too; which instances those are it says rightly but for one (bf16 in groups of 32 rows, three m-blocks of six n-tiles: 249).
constexpr int regs_estimate(int mb, int j, int sub, bool w8) {
  const int pl = w8 ? 2 : 1;
  return 8 * j * pl + 4 * j * mb + 16 * mb + 4 * pl * mb + (4 + sub) * mb + (sub == 4 ? 65 : 45);
}
// Launch shapes: eight wavefronts for up to four n-tiles, four for three to eight (of 8-bit codes to six), up to three m-blocks (8-bit codes in
// groups of 32 rows, three m-blocks of four n-tiles: more registers than eight wavefronts have).
constexpr bool regs_built(int mb, int j, int nw, int sub, bool w8) {
  return mb >= 1 && mb <= 3 && (nw == 8 ? j >= 1 && j <= 4 && !(w8 && sub == 4 && mb * j == 12) : nw == 4 && j >= 3 && j <= (w8 ? 6 : 8));
}

template <bool BF16, bool HAS_ZP, int SUBG, bool W8, int NW, int J, int MB, int MR = 16>
static int launch_regs(const RegsParams& p, hipStream_t s) {
  if constexpr (MB == 1 && MR == 16)
    if (p.M <= 4) return launch_regs<BF16, HAS_ZP, SUBG, W8, NW, J, MB, 4>(p, s);
  constexpr size_t lds = regs_lds_bytes(MB, MR, J, NW, SUBG, HAS_ZP);
  static_assert(lds <= 160 * 1024, "LDS");
  auto kern = w4a16_regs_kernel<BF16, MB, MR, J, HAS_ZP, NW, SUBG, W8, NW == 4 && (regs_estimate(MB, J, SUBG, W8) > 256) ? 1 : 2>;
  static size_t reserved[VAQ_MAX_DEVICES];
  if (const int rc = reserve_dynamic_lds(reinterpret_cast<const void*>(kern), lds, reserved, "w4a16_gemm(regs)"); rc != VAQ_OK) return rc;
  const KernelHead h = regs_head(p);
  hipLaunchKernelGGL(kern, dim3(p.per_xcd * 8), dim3(NW * 64), lds, s, h.a, h.b, h.c, p);
  return VAQ_OK;
}

template <bool BF16, bool HAS_ZP, int SUBG, bool W8, int NW, int J = 1>
static int regs_dispatch(const RegsParams& p, int j, int mb, hipStream_t s) {
  if constexpr (J > 8) {
    set_error("w4a16_gemm(regs): %d n-tiles and %d m-blocks on %d wavefronts are not built", j, mb, NW);
    return VAQ_ERR_UNSUPPORTED;
  } else {
    if constexpr (regs_built(1, J, NW, SUBG, W8))
      if (j == J && mb == 1) return launch_regs<BF16, HAS_ZP, SUBG, W8, NW, J, 1>(p, s);
    if constexpr (regs_built(2, J, NW, SUBG, W8))
      if (j == J && mb == 2) return launch_regs<BF16, HAS_ZP, SUBG, W8, NW, J, 2>(p, s);
    if constexpr (regs_built(3, J, NW, SUBG, W8))
      if (j == J && mb == 3) return launch_regs<BF16, HAS_ZP, SUBG, W8, NW, J, 3>(p, s);
    return regs_dispatch<BF16, HAS_ZP, SUBG, W8, NW, J + 1>(p, j, mb, s);
  }
}

template <int SUBG, bool W8, bool HAS_ZP>
static int regs_types(const RegsParams& p, int nw, int j, int mb, bool bf16, hipStream_t s) {
  if (nw == 8) return bf16 ? regs_dispatch<true, HAS_ZP, SUBG, W8, 8>(p, j, mb, s) : regs_dispatch<false, HAS_ZP, SUBG, W8, 8>(p, j, mb, s);
  return bf16 ? regs_dispatch<true, HAS_ZP, SUBG, W8, 4>(p, j, mb, s) : regs_dispatch<false, HAS_ZP, SUBG, W8, 4>(p, j, mb, s);
}

// One file each (w4a16_regs_*.hip): 4-bit codes in groups of 128 / 64 / 32 rows, 8-bit codes likewise.
int regs_launch_w4(const RegsParams& p, int nw, int j, int mb, bool bf16, bool zp, hipStream_t s);
int regs_launch_w4_sub2(const RegsParams& p, int nw, int j, int mb, bool bf16, bool zp, hipStream_t s);
int regs_launch_w4_sub4(const RegsParams& p, int nw, int j, int mb, bool bf16, bool zp, hipStream_t s);
int regs_launch_w8(const RegsParams& p, int nw, int j, int mb, bool bf16, hipStream_t s);
int regs_launch_w8_sub2(const RegsParams& p, int nw, int j, int mb, bool bf16, hipStream_t s);
int regs_launch_w8_sub4(const RegsParams& p, int nw, int j, int mb, bool bf16, hipStream_t s);

}  // namespace vaq
