// FP8 GEMM for some dozen rows: the K loop of w4a16_regs_kernel.h without codes to unpack and scales to apply.
//
//  * A wavefront multiplies one step of 256 bytes of K of MB * 16 rows with J neighbouring n-tiles; the wavefronts of a workgroup take a quarter of K each and
//    share nothing until their sums meet in LDS at the end: no barrier in the K loop, no hand-over between workgroups, no scratch.
//  * Activations and weights come by direct-to-LDS loads of 4 rows x 256 contiguous bytes into a piece of LDS of the wavefront's own, weights two steps ahead,
//    activations one.
//  * Rows beyond MB * 16 are a further block of rows with workgroups of their own, side by side on the same XCD, so that they find the weights in its L2.
//
// What bounds the kernels that took these calls: the stream kernels load every row's share of K into registers in the operand layout, 16 rows x 64 bytes an
// instruction, ahead of the first product (2 us for each 16 rows of K = 4096), and the tile kernels run 64 rows and more on a quarter of the device or hand partial
// tiles over, 0.27 us for a step of 128 bytes.  What bounds this one: the bytes that pass into a compute unit, MB + J tiles a step at 45 B/ns.
// Cold, us, before -> now: 2048 x 2048 at M = 32 / 64 4.2 / 6.7 -> 3.2 / 3.7; 4096 x 4096 at M = 32 / 64 / 128 7.6 / 10.0 / 10.0 -> 6.0 / 6.9 / 8.6; 4096 x 6144 at
// M = 64 10.4 -> 8.5; 11008 x 4096 at M = 32 14.6 -> 12.1; 2560 x 1280 at M = 64 8.2 -> 4.2.
// Not kept: weights straight into registers in the operand layout (16 rows x 64 bytes an instruction pass at 25 B/ns: 2048 x 2048 at M = 64 4.6, 4096 x 4096 8.8 us, in
// either order of a lane's two halves), steps of 128 bytes (3.9, 7.3) or eight wavefronts (4.1, 7.1), activations as far ahead as weights and three or four steps
// ahead (4.1, 7.4).
#pragma once
#include "fp8_stream2_kernel.h"

namespace vaq {

constexpr int FP8_REGS_WAVES = 4, FP8_REGS_STEP = 256;
constexpr size_t fp8_regs_lds_bytes(int mb, int j) {
  const size_t run = (size_t)FP8_REGS_WAVES * (mb + 2 * j) * 16 * FP8_REGS_STEP, sums = (size_t)FP8_REGS_WAVES * j * mb * 1024;
  return run > sums ? run : sums;
}

// What a workgroup computes: a range of n-tiles and a block of rows; the row blocks of a range are neighbours on one XCD.  unit / RB by multiplication: exact for
// unit * RB < 2^32.  (Callable on the host for its test.)
inline uint32_t fp8_regs_magic(uint32_t RB) { return (uint32_t)((1ull << 32) / RB + 1); }
struct Fp8RegsUnit {
  uint32_t range, rb;
};
__host__ __device__ inline uint32_t fp8_regs_place(uint32_t block, uint32_t per_xcd) { return (block & 7u) * per_xcd + (block >> 3); }
__host__ __device__ inline Fp8RegsUnit fp8_regs_unit(uint32_t unit, uint32_t RB, uint32_t magic) {
  Fp8RegsUnit u{unit, 0};
  if (RB > 1) {
    u.range = mul_high(unit, magic);
    u.rb = unit - u.range * RB;
  }
  return u;
}

// TAIL: K ends inside a step.  What a row has behind K is not its own (a NaN in the weights is one whatever it is multiplied with): of the last step each lane asks
// for the chunks before K, and the rest of both operands arrives as zeros.
template <bool BF16_OUT, int MB, int J, bool TAIL>
__global__ __launch_bounds__(FP8_REGS_WAVES * 64, 2) void fp8_mm_regs_kernel(VAQ_HEAD_ARGS, const Fp8MMParams p) {
  using T = F16Traits<BF16_OUT>;
  constexpr int NW = FP8_REGS_WAVES, KT = FP8_REGS_STEP, R = (J * MB + NW - 1) / NW, TB = 16 * KT, LI = TB / 1024;
  const uint8_t* const a = head_ptr<uint8_t>(h0[0], h0[1]);
  const uint8_t* const b = head_ptr<uint8_t>(h0[2], h0[3]);
  const uint32_t lda = h0[4], ldb = h0[5], a_extent = h0[6], b_extent = h0[7];
  const int all = (int)(h1[0] >> 8), rest = (int)(h1[0] & 0xffu), M = (int)(h1[1] & 0xffffu), NT = (int)h2[0];
  const uint32_t RB = h1[1] >> 16, ranges = h1[2], per_xcd = h1[3];
  extern __shared__ __attribute__((aligned(16))) uint8_t lds8[];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int q = lane >> 4, r16 = lane & 15;
  const uint32_t unit = fp8_regs_place(blockIdx.x, per_xcd);
  if (unit >= ranges * RB) return;
  const Fp8RegsUnit u = fp8_regs_unit(unit, RB, h2[1]);
  const uint32_t range = u.range, rb_u = u.rb;
  const int nt0 = (int)range * J, row0 = (int)rb_u * MB * 16;

  // steps first .. steps - 1 of K are this wavefront's
  const int per = (all + NW - 1) / NW, first = w * per, steps = min(first + per, all);

  auto rsrc = [](const void* base, uint32_t bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000); };
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  uint8_t* const mine = lds8 + (size_t)w * ((MB + 2 * J) * TB);
  // a load instruction fetches four whole rows of a tile of 16; their 16-byte chunk c is at place c ^ row: the 16 rows of an operand read hit all banks
  uint32_t vo_a[LI * MB], vo_w[LI];
#pragma unroll
  for (int i = 0; i < LI * MB; ++i) {
    const int r = i * 4 + q;
    vo_a[i] = (uint32_t)min(row0 + r, M - 1) * lda + (uint32_t)((r16 ^ (r & 15)) * 16);
  }
#pragma unroll
  for (int i = 0; i < LI; ++i) {
    const int r = i * 4 + q;
    vo_w[i] = (uint32_t)r * ldb + (uint32_t)((r16 ^ r) * 16);
  }
  // A step past the last has no extent and starts at 0 (vaq_common.h): its requests fetch nothing and keep the count of requests under way.
  auto place = [&](uint32_t vo, int r, int g) {
    if constexpr (TAIL) return g == all - 1 && ((r16 ^ (r & 15)) * 16) >= rest ? 0x80000000u : vo;
    return vo;
  };
  auto load_act = [&](int g) {
    const __amdgpu_buffer_rsrc_t ra = rsrc(a, g < steps ? a_extent : 0u);
#pragma unroll
    for (int i = 0; i < LI * MB; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(mine + i * 1024), 16, (int)place(vo_a[i], i * 4 + q, g), g < steps ? g * KT : 0, 0, 0);
  };
  auto load_w = [&](int s, int g) {
    const __amdgpu_buffer_rsrc_t rb = rsrc(b, g < steps ? b_extent : 0u);
#pragma unroll
    for (int j = 0; j < J; ++j) {
      const int so = g < steps ? (int)((uint32_t)(min(nt0 + j, NT - 1) * 16) * ldb + (uint32_t)(g * KT)) : 0;
#pragma unroll
      for (int i = 0; i < LI; ++i)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_ptr_t)(mine + (MB + s * J + j) * TB + i * 1024), 16, (int)place(vo_w[i], i * 4 + q, g), so, 0, 2);
    }
  };
  v4f acc[J][MB];
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[j][mb] = v4f{0.f, 0.f, 0.f, 0.f};

  auto operand = [&](const uint8_t* at, int u) {
    const v4i lo = *reinterpret_cast<const v4i*>(at + r16 * KT + ((u * 8 + q) ^ r16) * 16);
    const v4i hi = *reinterpret_cast<const v4i*>(at + r16 * KT + ((u * 8 + 4 + q) ^ r16) * 16);
    return v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
  };
  constexpr int U = KT / 128;
  auto tile = [&](int s, bool refill_act, bool refill_w, int next_act, int next_w) {
    v8i act[U][MB], wop[U][J];
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) act[u][mb] = operand(mine + mb * TB, u);
#pragma unroll
      for (int j = 0; j < J; ++j) wop[u][j] = operand(mine + (MB + s * J + j) * TB, u);
    }
    if (refill_act) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // this step's are in registers
      __builtin_amdgcn_sched_barrier(0);
      load_act(next_act);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (refill_w) {
      load_w(s, next_w);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int j = 0; j < J; ++j)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[j][mb] = mfma_fp8_16(wop[u][j], act[u][mb], acc[j][mb]);
  };

  // W(0) A(0) W(1) | A(1) W(2) | A(2) W(3) | ..., `|` = a step: it starts when all but the weights requested behind its activations have been answered
  auto wait = [&] { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(J * LI) : "memory"); };
  int g = first;
  load_w(0, g);
  __builtin_amdgcn_sched_barrier(0);
  load_act(g);
  __builtin_amdgcn_sched_barrier(0);
  if (g + 1 < steps) load_w(1, g + 1);
  __builtin_amdgcn_sched_barrier(0);
  VAQ_ARRIVED4(p.sb, p.bias, p.out, p.sb_per_col);
  const __amdgpu_buffer_rsrc_t rsa = rsrc(p.sa, p.sa_per_row ? (uint32_t)M * 4u : 4u), rsb = rsrc(p.sb, p.sb_per_col ? (uint32_t)NT * 64u : 4u),
                               rbias = rsrc(p.bias, p.bias ? (uint32_t)NT * 32u : 0u);
  // Scales and bias of this wavefront's results, ahead of the K loop (behind it they are a round trip to memory on their own).  Two loads for each result, which a lone step's wait
  // counts: the compiler merges none of them, because it cannot see their offsets.  One scale for all columns is the first of four and is spread where it is used: here that would
  // wait for all requests (1024 x 21584 at M = 14 7.6 -> 6.6 us, 261 drawn calls with one scale 0.971).
  v4f sb4[R];
  v2u bias4[R];
  float sam[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int u = w + i * NW, j = u / MB, mb = u - j * MB, n = min(nt0 + j, NT - 1) * 16 + q * 4, m = min(row0 + mb * 16 + r16, M - 1);
    int at[3] = {p.sa_per_row ? m * 4 : 0, p.sb_per_col ? n * 4 : 0, n * 2};
#ifdef __HIP_DEVICE_COMPILE__
    asm volatile("" : "+v"(at[0]), "+v"(at[1]), "+v"(at[2])::"memory");
#endif
    sam[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsa, at[0], 0, 0));
    sb4[i] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rsb, at[1], 0, 0));
    bias4[i] = v2u{0u, 0u};
    if (p.bias) bias4[i] = __builtin_bit_cast(v2u, __builtin_amdgcn_raw_buffer_load_b64(rbias, at[2], 0, 0));
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll 1
  for (; g + 2 < steps; g += 2) {
    wait();
    tile(0, true, true, g + 1, g + 2);
    wait();
    tile(1, true, true, g + 2, g + 3);
  }
  // the last one or two ask for no weights (requests for nothing behind them cost 3 % of a call)
  if (g + 1 < steps) {
    wait();
    tile(0, true, false, g + 1, 0);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    tile(1, false, false, 0, 0);
  } else if (g < steps) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * R) : "memory");      // (all but the scales)
    tile(0, false, false, 0, 0);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // (what is requested past the end writes zeros into LDS)

  v4f* const red = reinterpret_cast<v4f*>(lds8);      // [NW][J * MB][64], on top of the activations
  __syncthreads();
#pragma unroll
  for (int j = 0; j < J; ++j)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) red[(w * (J * MB) + j * MB + mb) * 64 + lane] = acc[j][mb];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int u = w + i * NW, j = u / MB, mb = u - j * MB, nt = nt0 + j, m = row0 + mb * 16 + r16;
    if (u >= J * MB || nt >= NT) continue;
    v4f val = red[u * 64 + lane];
#pragma unroll
    for (int ww = 1; ww < NW; ++ww) val += red[(ww * (J * MB) + u) * 64 + lane];
    if (m < M) {
#pragma clang fp contract(off)      // sa * (sb * acc), then + bias: two fp32 roundings, like the tile kernels
      const uint16_t bias_r[4] = {(uint16_t)(bias4[i].x & 0xffffu), (uint16_t)(bias4[i].x >> 16), (uint16_t)(bias4[i].y & 0xffffu), (uint16_t)(bias4[i].y >> 16)};
      float o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        o[r] = sam[i] * ((p.sb_per_col ? sb4[i][r] : sb4[i][0]) * val[r]);
        if (p.bias) o[r] += T::to_float(bias_r[r]);
      }
      v2u ov;
      ov.x = (uint32_t)T::from_float(o[0]) | ((uint32_t)T::from_float(o[1]) << 16);
      ov.y = (uint32_t)T::from_float(o[2]) | ((uint32_t)T::from_float(o[3]) << 16);
      *reinterpret_cast<v2u*>(p.out + (int64_t)m * p.ldc + nt * 16 + q * 4) = ov;
    }
  }
}

constexpr bool fp8_regs_built(int mb, int j) { return mb >= 1 && mb <= 4 && j >= 1 && j <= 4 && fp8_regs_lds_bytes(mb, j) <= 160 * 1024; }
constexpr int FP8_REGS_MAX_M = 256;
// The cheapest plan of a problem and its predicted time.
struct Fp8RegsPlan {
  int mb = 0, j = 0;
  double us = -1;
};
Fp8RegsPlan fp8_regs_plan(int M, int N, int K);
// false: not built, or no room in LDS
bool fp8_regs_launch(const Fp8MMParams& p, bool bf16, int mb, int j, hipStream_t s);

}  // namespace vaq
