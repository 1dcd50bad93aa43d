// The FP8 GEMM for few rows whose weights pass through LDS, and the parameters that all FP8 GEMM kernels share.
#pragma once
#include "tile_handover.h"
#include "vaq_common.h"

#include <type_traits>

namespace vaq {

struct Fp8MMParams {
  const uint8_t* a;
  int64_t lda;
  const uint8_t* b;
  int64_t ldb;
  const float* sa;
  int sa_per_row;   // 1: sa[m], 0: sa[0]
  const float* sb;
  int sb_per_col;
  const uint16_t* bias;
  uint16_t* out;
  int64_t ldc;
  int M, N, K;
  float* c_tmp = nullptr;        // fp32 partial tiles when K is split over workgroups (SK > 1)
  int32_t* counters = nullptr;   // arrival counters, zero on entry, left zero
  int SK = 1;
  int tail_first = 0;            // 0: every tile in SK parts; > 0: only the tiles from this position on (see tile_slot)
  int rotate_k = 0;              // multi-stage tile kernel: 1 tile rows, 2 tile columns start their K loop at different places (see the kernel)
  int m_tiles_extra = 0;         // multi-stage tile kernel: tile rows past M (see dispatch_tile: they read the weights with the real ones and store nothing)
  uint32_t a_extent = 0, b_extent = 0;   // bytes up to the end of the last row of a / b (stream kernels: below 2 GiB, tile kernels 4)
  TileSplitMagic split_magic = {0, 0};      // see tile_handover.h
  uint32_t rotate_magic = 0;     // of the tile rows (rotate_k = 1) or columns (2)
  int nt_base = 0, nt_rem = 0;   // stream kernel: n-tiles per workgroup = nt_base, one more for the first nt_rem (N/16 split on the host)
};

__device__ inline v4f mfma_fp8_16(v8i a, v8i b, v4f c) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
}

// The maxima of MQ registers over the 64 lanes (no LDS): lane l gets that of register l mod MQ.  A swap of half wavefronts
// and a maximum fold two registers into one, twice; the rest is a rotation inside the rows of 16 lanes.
template <int MQ>
static __device__ inline uint32_t wave_maxima(uint32_t (&v)[MQ]) {
  auto ror = [](uint32_t x) {
    x = max(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x128, 0xf, 0xf, true));      // row_ror:8, 4, 2, 1
    x = max(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x124, 0xf, 0xf, true));
    x = max(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x122, 0xf, 0xf, true));
    return max(x, (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0x121, 0xf, 0xf, true));
  };
  auto fold32 = [](uint32_t a, uint32_t b) {      // lanes 0 .. 31: of a, 32 .. 63: of b
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    return max(r[0], r[1]);
  };
  auto fold16 = [](uint32_t a, uint32_t b) {      // even rows of 16 lanes: of a, odd rows: of b
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    return max(r[0], r[1]);
  };
  const int lane = threadIdx.x;
  if constexpr (MQ == 1) {
    const uint32_t x = ror(v[0]), y = fold16(x, x);
    return fold32(y, y);
  } else if constexpr (MQ == 2) {
    const uint32_t x = ror(fold32(v[0], v[1])), y = fold16(x, x);      // a half wavefront each
    return (uint32_t)__builtin_amdgcn_ds_bpermute((lane & 1) * 128, (int)y);
  } else {
    // register j of MQ / 4: row of lanes (half, row) holds v[half * MQ / 2 + row * MQ / 4 + j]
    uint32_t out = 0;
    uint32_t x[MQ / 4];
#pragma unroll
    for (int j = 0; j < MQ / 4; ++j) {
      const uint32_t a = fold32(v[j], v[MQ / 2 + j]), b = fold32(v[MQ / 4 + j], v[MQ / 2 + MQ / 4 + j]);
      x[j] = ror(fold16(a, b));
    }
    const int want = lane & (MQ - 1), src = ((want / (MQ / 2)) * 32 + ((want / (MQ / 4)) & 1) * 16) * 4;
#pragma unroll
    for (int j = 0; j < MQ / 4; ++j) {
      const uint32_t t = (uint32_t)__builtin_amdgcn_ds_bpermute(src, (int)x[j]);
      out = (want & (MQ / 4 - 1)) == j ? t : out;
    }
    return out;
  }
}

// What the first requests of the stream kernels need, as their head (vaq_common.h); the rest is loaded.
__device__ inline Fp8MMParams stream_params(const v8u& h0, const v4u& h1, const v2u& h2, const Fp8MMParams& rest) {
  Fp8MMParams p = rest;
  p.a = head_ptr<uint8_t>(h0[0], h0[1]);
  p.b = head_ptr<uint8_t>(h0[2], h0[3]);
  p.sa = head_ptr<float>(h0[4], h0[5]);
  p.lda = h0[6];
  p.ldb = h0[7];
  p.K = (int)h1[0];
  p.M = (int)(h1[1] & 0xffffu);
  p.a_extent = h1[2];
  p.b_extent = h1[3];
  p.nt_base = (int)h2[0];
  p.nt_rem = (int)h2[1];
  return p;
}
template <class Kernel>
inline void launch_fp8_stream(Kernel kern, dim3 grid, int wk, size_t lds, hipStream_t s, const Fp8MMParams& p) {
  hipLaunchKernelGGL(kern, grid, dim3(64, wk), lds, s,
                     (v8u{ptr_lo(p.a), ptr_hi(p.a), ptr_lo(p.b), ptr_hi(p.b), ptr_lo(p.sa), ptr_hi(p.sa), (uint32_t)p.lda, (uint32_t)p.ldb}),
                     (v4u{(uint32_t)p.K, (uint32_t)p.M | (uint32_t)wk << 16, p.a_extent, p.b_extent}), (v2u{(uint32_t)p.nt_base, (uint32_t)p.nt_rem}), p);
}

// ----------------------------------------------------------------------------- stream kernel, weights through LDS
// fp8_mm_stream_kernel (fp8_scaled_mm.hip) fetches the weights in the MFMA operand layout: every load instruction takes
// 64-byte pieces of 16 rows, half a cache line each.  Measured on bare reads of a 4096 x 28672 byte matrix with cold lines, that
// pattern reaches 4.2-5.3 TB/s where instructions that read whole lines reach 5.3-5.9 TB/s.  Here every load
// instruction is a direct-to-LDS load of 4 rows x 256 contiguous bytes into a ring that belongs to the wavefront alone
// (no barrier: the wavefront waits on its own load counter), and the operands are read back from LDS, 16-byte chunks
// XOR-swizzled by the row so that the 16 rows of an operand read hit 16 different bank groups.
//  * blockDim = (64, WK).  Wavefront w owns K steps [w*KS, (w+1)*KS) of 128 bytes; its activations live in registers;
//    the workgroup walks a contiguous range of 16-row n-tiles; per n-tile the wavefronts reduce through LDS as there.
//  * A stage is two steps (16 rows x 256 bytes = 4 KiB, four load instructions); the ring holds NSR stages, and the
//    stage NSR ahead -- of this n-tile or the next -- is requested as soon as a stage's operands have been read.
//  * MQ > 0: the activations come as the 16-bit numbers they are before their quantisation (type BF16_OUT, at most MQ rows),
//    and every wavefront quantises its own K slab, bit for bit as the quantisation kernels do: per token (p.sa null) or with
//    the one scale at p.sa (STATIC).  A layer is then one launch instead of two.
template <bool BF16_OUT, int KS, int MB, int NSR, int MQ = 0, bool STATIC = false>
__global__ __launch_bounds__(512) void fp8_mm_stream2_kernel(VAQ_HEAD_ARGS, const Fp8MMParams rest) {
  const Fp8MMParams p = stream_params(h0, h1, h2, rest);
  const int WK = (int)(h1[1] >> 16);
  using T = F16Traits<BF16_OUT>;
  constexpr int NS = KS / 2;                       // stages per n-tile
  static_assert(KS % 2 == 0 && NS % NSR == 0, "whole stages, ring slots fixed at compile time");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds8[];
  const int lane = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.y);
  const int q = lane >> 4, r16 = lane & 15;
  const int kw = w * KS * 128;                     // first byte of K of this wavefront
  const int kbase = kw + q * 32;
  uint8_t* const ring = lds8 + (size_t)w * NSR * 4096;
  v4f* const red = reinterpret_cast<v4f*>(lds8 + (size_t)WK * NSR * 4096);      // [2][WK][MB][64]

  constexpr uint32_t OOB = 0x80000000u;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.a), 0, (int)p.a_extent, 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.b), 0, (int)p.b_extent, 0x00020000);
  v8i breg[KS][MB];
  // 16-bit activations of the wavefront's K slab: register i = (row i / PARTS, numbers 512 (i % PARTS) + 8 lane .. + 7)
  constexpr int PARTS = KS / 4;
  static_assert(MQ == 0 || (MB == 1 && KS % 4 == 0), "quantised here: one m-block, whole pieces of 512 numbers");
  v4u raw[MQ > 0 ? MQ * PARTS : 1];
  if constexpr (MQ > 0) {
#pragma unroll
    for (int i = 0; i < MQ * PARTS; ++i) {
      const int m = i / PARTS, k = kw + (i % PARTS) * 512 + lane * 8;
      const uint32_t off = (m < p.M && k < p.K) ? ((uint32_t)m * (uint32_t)p.lda + (uint32_t)k) * 2u : OOB;
      raw[i] = __builtin_amdgcn_raw_buffer_load_b128(ra, (int)off, 0, 0);
    }
  }
#pragma unroll
  for (int s = 0; s < (MQ > 0 ? 0 : KS); ++s) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int m = mb * 16 + r16;
      const int k = kbase + s * 128;
      const uint32_t base = (uint32_t)m * (uint32_t)p.lda + (uint32_t)k;
      const uint32_t o_lo = (m < p.M && k < p.K) ? base : OOB, o_hi = (m < p.M && k + 16 < p.K) ? base + 16u : OOB;
      const v4i lo = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(ra, (int)o_lo, 0, 0));
      const v4i hi = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(ra, (int)o_hi, 0, 0));
      breg[s][mb] = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    }
  }

  const int NT = p.N / 16;
  const int bx = blockIdx.x;
  const int nt0 = bx * p.nt_base + (bx < p.nt_rem ? bx : p.nt_rem);
  const int nt1 = nt0 + p.nt_base + (bx < p.nt_rem ? 1 : 0);

  // Load instruction i of a stage fills LDS bytes [1024 i, 1024 i + 1024) = rows 4i .. 4i+3; lane l lands at row
  // 4i + l/16, position l & 15, which holds chunk (l & 15) ^ row of the row's 256 bytes.
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  uint32_t voffb[4], kchunk[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 4 * i + (lane >> 4);
    kchunk[i] = (uint32_t)(((lane & 15) ^ row) * 16);
    voffb[i] = (uint32_t)row * (uint32_t)p.ldb + kchunk[i];
  }
  // `live` = false requests nothing (offsets beyond the extent) but keeps the count of loads in flight the same, and so does a stage past K.  (The scalar offset stays in the
  // operand: vaq_common.h.)
  uint32_t k_at[NS];
#pragma unroll
  for (int st = 0; st < NS; ++st) k_at[st] = (uint32_t)min(kw + st * 256, p.K);
  auto rows_of = [&](int nt) { return (uint32_t)(max(min(nt, nt1 - 1), 0) * 16) * (uint32_t)p.ldb; };
  auto issue_stage = [&](uint32_t rows, int st, int slot, bool live) {
    const int k0 = kw + st * 256;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t vo = (live && k0 + (int)kchunk[i] < p.K) ? voffb[i] : OOB;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_ptr_t)(ring + slot * 4096 + i * 1024), 16, (int)vo, (int)(rows + k_at[st]), 0, 2);
    }
  };
#pragma unroll
  for (int st = 0; st < NSR; ++st) issue_stage(rows_of(nt0), st, st, nt0 < nt1);
  // (M = 16 on 4096 x 6144 7.08 -> 6.88 us, M = 7 on 4096 x 4096 5.36 -> 5.07, 5.21 with the wait ahead of the loop below.  Quantised here it is there: a given
  // scale's own load would come behind it, 4096 x 6144 at M = 8 7.02 -> 8.02.)
  if constexpr (MQ == 0) VAQ_ARRIVED4(p.sb, p.bias, p.out, p.sb_per_col);

  const bool reducer_wave = WK > 1 ? w < MB : true;
  float sam_mb[MB];
  if constexpr (MQ > 0) {
    float s;                            // per token: lane l holds the scale of row l mod MQ
    const int mr = lane & (MQ - 1);
    if constexpr (STATIC) {
      s = *p.sa;
    } else {
      // the magnitudes on the bits, two numbers an operation: 2x + TOP drops the sign and orders numbers at TOP and above,
      // NaNs (which count for nothing) below
      typedef uint16_t v2us __attribute__((ext_vector_type(2)));
      constexpr uint16_t TOP = BF16_OUT ? 0x00ff : 0x07ff;
      uint32_t tops[MQ];
#pragma unroll
      for (int m = 0; m < MQ; ++m) {
        v2us v = {TOP, TOP};
#pragma unroll
        for (int i = m * PARTS; i < (m + 1) * PARTS; ++i) {
          const uint32_t x[4] = {raw[i].x, raw[i].y, raw[i].z, raw[i].w};
#pragma unroll
          for (int e = 0; e < 4; ++e) v = __builtin_elementwise_max(v, (v2us)(__builtin_bit_cast(v2us, x[e]) * (v2us){2, 2} + (v2us){TOP, TOP}));
        }
        tops[m] = max((uint32_t)v.x, (uint32_t)v.y);
      }
      uint32_t top = wave_maxima<MQ>(tops);
      if (WK > 1) {
        // (in the half of the reduction buffer that nobody writes before every wavefront has read this)
        uint32_t* const part = reinterpret_cast<uint32_t*>(red + (size_t)WK * MB * 64);
        if (lane < MQ) part[w * MQ + lane] = top;
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        uint32_t t[8];
#pragma unroll
        for (int ww = 0; ww < 8; ++ww) t[ww] = part[min(ww, WK - 1) * MQ + mr];
#pragma unroll
        for (int ww = 0; ww < 8; ++ww) top = max(top, t[ww]);
      }
      s = fmaxf(T::to_float((uint16_t)((top - TOP) >> 1)) / 448.0f, 1.0f / (448.0f * 512.0f));
    }
    const float rcp = 1.0f / s;
    // Quotients as in fp8_quant.hip.  A scale of infinity (a row with one): 0 in the place of s leaves q = x * 0, the same
    // quotient, and the correction steps of div16_exact then change nothing.
    const float s_div = s < __builtin_inff() ? s : 0.f;
    uint8_t* const stage = lds8 + (size_t)WK * NSR * 4096 + (WK > 1 ? (size_t)2 * WK * MB * 1024 : 0) + (size_t)w * MQ * 128;
    v2u code[MQ * PARTS];
#pragma unroll
    for (int i = 0; i < MQ * PARTS; ++i) {
      const int m = i / PARTS;
      const float s_m = STATIC ? s_div : __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, s_div), m));
      const float r_m = STATIC ? rcp : __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, rcp), m));
      auto quot = [&](uint32_t h) {
        // The steps of div16_exact, which is inline assembly: in front of that the compiler fills in wait states, a third of
        // the instructions here.  (Per token the magnitude is at most 448 up to the last bit, which the conversion rounds
        // away: only a NaN needs the minimum.)
        const float x = T::to_float((uint16_t)h), qu = x * r_m;
        float y = qu;
        if constexpr (!STATIC) {
          const float e = __builtin_fmaf(qu, s_m, -x);
          y = __builtin_fmaf(-e, r_m, qu);
        }
        y = fminf(y, 448.0f);
        if constexpr (STATIC) y = fmaxf(-448.0f, y);
        return y;
      };
      const uint32_t x[4] = {raw[i].x, raw[i].y, raw[i].z, raw[i].w};
      int c[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        c[h] = __builtin_amdgcn_cvt_pk_fp8_f32(quot(x[2 * h] & 0xffffu), quot(x[2 * h] >> 16), 0, false);
        c[h] = __builtin_amdgcn_cvt_pk_fp8_f32(quot(x[2 * h + 1] & 0xffffu), quot(x[2 * h + 1] >> 16), c[h], true);
      }
      code[i] = v2u{(uint32_t)c[0], (uint32_t)c[1]};
    }
    // The codes reach the operand layout through a piece of LDS of this wavefront alone, a step of 128 codes of every row at
    // a time (its LDS operations run in order).  Two rows are one 256-byte line, 16-byte chunks XOR-ed by the line.
    // (Columns past MQ of the product are never stored.)
    auto at = [&](int m, int c) { return stage + (m >> 1) * 256 + ((((m & 1) * 8 + c) ^ (m >> 1)) * 16); };
#pragma unroll
    for (int st = 0; st < KS; ++st) {
      if ((lane >> 4) == (st & 3)) {
#pragma unroll
        for (int m = 0; m < MQ; ++m) *reinterpret_cast<v2u*>(at(m, r16 >> 1) + (r16 & 1) * 8) = code[m * PARTS + st / 4];
      }
      asm volatile("" ::: "memory");
      const v4i lo = *reinterpret_cast<const v4i*>(at(mr, 2 * q)), hi = *reinterpret_cast<const v4i*>(at(mr, 2 * q + 1));
      breg[st][0] = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      asm volatile("" ::: "memory");
    }
    sam_mb[0] = s;
  }
#pragma unroll
  for (int mb = 0; mb < (MQ > 0 ? 0 : MB); ++mb) {
    const int m = mb * 16 + r16;
    sam_mb[mb] = (reducer_wave && m < p.M) ? p.sa[p.sa_per_row ? m : 0] : 0.f;
  }

  const __amdgpu_buffer_rsrc_t rsb =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.sb), 0, p.sb_per_col ? p.N * 4 : 4, 0x00020000);
  const __amdgpu_buffer_rsrc_t rbias =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p.bias), 0, p.bias ? p.N * 2 : 0, 0x00020000);
  if constexpr (MQ > 0) VAQ_ARRIVED4(p.sb, p.bias, p.out, p.sb_per_col);
  int parity = 0;
  for (int nt = nt0; nt < nt1; ++nt) {
    v4f acc[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[mb] = v4f{0.f, 0.f, 0.f, 0.f};
    // the tile's weight scales and bias, by every wavefront and without a branch (a missing bias has no extent and reads as
    // zeros): the waits below count on two requests here, and a wait of their own would drain the ring
    const v4f sb4 = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rsb, p.sb_per_col ? (nt * 16 + q * 4) * 4 : 0, 0, 0));
    const v2u bias4 = __builtin_bit_cast(v2u, __builtin_amdgcn_raw_buffer_load_b64(rbias, (nt * 16 + q * 4) * 2, 0, 0));
    asm volatile("" ::: "memory");
#pragma unroll
    for (int st = 0; st < NS; ++st) {
      // load instructions requested after this stage's (any others in flight only make the wait stricter)
      if (st < NSR) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NSR - 1) * 4 + 2) : "memory");
      else asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NSR - 1) * 4) : "memory");
      const int slot = st % NSR;
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        const int c0 = 8 * s2 + 2 * q;
        const v4i lo = *reinterpret_cast<const v4i*>(ring + slot * 4096 + r16 * 256 + ((c0 ^ r16) << 4));
        const v4i hi = *reinterpret_cast<const v4i*>(ring + slot * 4096 + r16 * 256 + (((c0 + 1) ^ r16) << 4));
        const v8i aop = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[mb] = mfma_fp8_16(aop, breg[2 * st + s2][mb], acc[mb]);
      }
      // the slot is free once its operands are in registers: request the stage NSR ahead into it
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (st + NSR < NS) issue_stage(rows_of(nt), st + NSR, slot, true);
      else issue_stage(rows_of(nt + 1), st + NSR - NS, slot, nt + 1 < nt1);
    }

    v4f tot = v4f{0.f, 0.f, 0.f, 0.f};
    bool reducer = w < MB;
    if (WK > 1) {
      v4f* buf = red + (size_t)parity * WK * MB * 64;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) buf[(w * MB + mb) * 64 + lane] = acc[mb];
      // the partial tiles are written; the bare barrier leaves the next tile's weight requests in flight (a
      // __syncthreads() would wait for every direct-to-LDS load)
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      // up to eight parts, four or eight reads under way at a time (one by one each waits out the LDS latency, and the others wait for the reducer)
      auto sum = [&](auto most) {
        constexpr int N = decltype(most)::value;
        v4f part[N];
#pragma unroll
        for (int ww = 0; ww < N; ++ww) part[ww] = buf[(min(ww, WK - 1) * MB + w) * 64 + lane];
#pragma unroll
        for (int ww = 0; ww < N; ++ww)
          if (ww < WK) tot += part[ww];
      };
      if (reducer) {
        if (WK <= 4) sum(std::integral_constant<int, 4>{});
        else sum(std::integral_constant<int, 8>{});
      }
      parity ^= 1;
    } else {
      reducer = true;
    }
    if (reducer) {
      const int mb_lo = (WK > 1) ? w : 0, mb_hi = (WK > 1) ? w + 1 : MB;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        if (mb < mb_lo || mb >= mb_hi) continue;
        const v4f val = (WK > 1) ? tot : acc[mb];
        const int m = mb * 16 + r16;
        if (m < p.M) {
#pragma clang fp contract(off)      // sa * (sb * acc), then + bias: two fp32 roundings, like the tile kernels
          const int n = nt * 16 + q * 4;
          const uint16_t bias_r[4] = {(uint16_t)(bias4.x & 0xffffu), (uint16_t)(bias4.x >> 16), (uint16_t)(bias4.y & 0xffffu),
                                      (uint16_t)(bias4.y >> 16)};
          float o[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            o[r] = sam_mb[mb] * ((p.sb_per_col ? sb4[r] : sb4[0]) * val[r]);
            if (p.bias) o[r] += T::to_float(bias_r[r]);
          }
          v2u ov;
          ov.x = (uint32_t)T::from_float(o[0]) | ((uint32_t)T::from_float(o[1]) << 16);
          ov.y = (uint32_t)T::from_float(o[2]) | ((uint32_t)T::from_float(o[3]) << 16);
          *reinterpret_cast<v2u*>(p.out + (int64_t)m * p.ldc + n) = ov;
        }
      }
    }
  }
}

}  // namespace vaq
