// FP8 (e4m3fn x e4m3fn) scaled GEMM for gfx950:
//     out[m,n] = round( sa[m] * ( sb[n] * sum_k a[m,k] b[k,n] ) + bias[n] ),   fp32 accumulation and epilogue.
// a is [M,K] row-major, b is [K,N] column-major (= weight [N,K] row-major with row pitch ldb), so both operands are
// k-contiguous and go to the matrix cores without any data re-arrangement.
//
// The kernels:
//  * tile kernel (any M; fp8_mm_tile3_kernel): one workgroup of 4 or 8 wavefronts per BM x BN output tile, both operands by
//    direct-to-LDS loads through a ring of stages, v_mfma_f32_32x32x64_f8f6f4 (the full-rate gfx950 FP8 instruction, 32
//    bytes per lane per operand).  fp8_mm_tile_kernel, K in steps of 128 bytes through double-buffered, padded LDS
//    (pitch 144 B), takes what the multi-stage kernel cannot address;
//  * stream kernels (M <= 32; M <= 64 on narrow layers with K <= 4096): weight-streaming GEMV-like, weights are the A operand
//    of v_mfma_f32_16x16x128_f8f6f4, activations stay in registers, the wavefronts of a workgroup split K and reduce
//    through LDS; fp8_mm_stream2_kernel (fp8_stream2_kernel.h) brings the weights in through LDS as whole cache lines;
//  * fp8_mm_regs_kernel (fp8_regs_kernel.h; 5 .. 256 rows, where predicted ahead of the others): both operands as
//    whole lines through LDS that no other wavefront touches, several n-tiles and m-blocks a wavefront.
//
// The per-lane byte -> k assignment inside an MFMA operand is the same function for A and B, so any consistent choice
// of which 32 bytes a lane supplies yields the exact dot product; the tile and stream kernels give lane (row, q) the
// bytes k0 + 32*q .. k0 + 32*q + 31 of its row.
#include "vaq_common.h"
#include "fp8_regs_kernel.h"
#include "fp8_stream2_kernel.h"
#include "tile_handover.h"
#include "tile_plan.h"

#include <type_traits>

namespace vaq {

__device__ inline v16f mfma_fp8_32(v8i a, v8i b, v16f c) {
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, c, 0, 0, 0, 0, 0, 0);
}

constexpr int F8_BK = 128;       // bytes of K per step
constexpr int F8_PITCH = 144;    // LDS row pitch in bytes

// Epilogue of the tile kernels.  The MFMAs are issued with the weight fragment as the A operand, so a 32x32
// accumulator block holds D[n_local][m_local]: lane -> column m_local = lane & 31, registers e -> rows
// n_local = 8*(e/4) + 4*(lane/32) + e%4.  Four consecutive registers are four consecutive n of one output row: one
// 8-byte store, one scale load per row, one 16-byte load of the channel scales.
template <bool BF16_OUT, int WMB, int WNB>
__device__ inline void tile_epilogue(const Fp8MMParams& p, v16f (&acc)[WMB][WNB], int m0, int n0, int wm, int wn, int lane) {
#pragma clang fp contract(off)      // sa * (sb * acc), then + bias: two fp32 roundings, like the oracle's separate operations
  using T = F16Traits<BF16_OUT>;
  // Every scale and bias value this lane needs is requested before the first store: a load that follows a store to
  // memory it might alias cannot be moved above it, and the epilogue would pay one memory latency per 8-byte store.
  float sam[WMB];
#pragma unroll
  for (int i = 0; i < WMB; ++i) {
    const int m = m0 + wm * 32 * WMB + i * 32 + (lane & 31);
    sam[i] = m < p.M ? p.sa[p.sa_per_row ? m : 0] : 0.f;
  }
  v4f sbv[WNB][4];
  v2u bv[WNB][4];
#pragma unroll
  for (int j = 0; j < WNB; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int n = n0 + wn * 32 * WNB + j * 32 + 8 * q + 4 * (lane >> 5);
      sbv[j][q] = v4f{0.f, 0.f, 0.f, 0.f};
      bv[j][q] = v2u{0u, 0u};
      if (n < p.N) {
        if (p.sb_per_col) sbv[j][q] = *reinterpret_cast<const v4f*>(p.sb + n);
        else sbv[j][q] = v4f{p.sb[0], p.sb[0], p.sb[0], p.sb[0]};
        if (p.bias) bv[j][q] = *reinterpret_cast<const v2u*>(p.bias + n);
      }
    }
#pragma unroll
  for (int i = 0; i < WMB; ++i) {
    const int m = m0 + wm * 32 * WMB + i * 32 + (lane & 31);
    if (m >= p.M) continue;
    uint16_t* orow = p.out + (int64_t)m * p.ldc;
#pragma unroll
    for (int j = 0; j < WNB; ++j) {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int n = n0 + wn * 32 * WNB + j * 32 + 8 * q + 4 * (lane >> 5);
        if (n >= p.N) continue;
        float o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = sam[i] * (sbv[j][q][r] * acc[i][j][4 * q + r]);
        if (p.bias) {
          o[0] += T::to_float((uint16_t)(bv[j][q].x & 0xffffu));
          o[1] += T::to_float((uint16_t)(bv[j][q].x >> 16));
          o[2] += T::to_float((uint16_t)(bv[j][q].y & 0xffffu));
          o[3] += T::to_float((uint16_t)(bv[j][q].y >> 16));
        }
        v2u ov;
        ov.x = (uint32_t)T::from_float(o[0]) | ((uint32_t)T::from_float(o[1]) << 16);
        ov.y = (uint32_t)T::from_float(o[2]) | ((uint32_t)T::from_float(o[3]) << 16);
        *reinterpret_cast<v2u*>(orow + n) = ov;
      }
    }
  }
}

// Epilogue of the multi-stage kernel: same arithmetic as tile_epilogue, but the 16-bit results cross a wavefront-private
// piece of LDS (32 rows of WNB * 64 + 16 bytes) so that they leave as 16-byte stores, 8 or 16 lanes to a row.  With the
// direct 8-byte stores every instruction touches 32 rows with 16 bytes each, and the write requests of a whole device
// finishing its tiles at the same time (one 16-byte piece each) took 10-17 us per tile.
// Requires: every wavefront of the workgroup has finished reading the operand ring, out 16-byte aligned.
template <bool BF16_OUT, int WMB, int WNB>
__device__ inline void tile_epilogue_lds(const Fp8MMParams& p, v16f (&acc)[WMB][WNB], int m0, int n0, int wm, int wn, int lane,
                                         uint8_t* wave_lds) {
#pragma clang fp contract(off)      // sa * (sb * acc), then + bias: two fp32 roundings, like the oracle's separate operations
  using T = F16Traits<BF16_OUT>;
  constexpr int PITCH = WNB * 64 + 16;
  constexpr int CPR = WNB * 4;                 // 16-byte chunks per row
  float sam[WMB];
#pragma unroll
  for (int i = 0; i < WMB; ++i) {
    const int m = m0 + wm * 32 * WMB + i * 32 + (lane & 31);
    sam[i] = m < p.M ? p.sa[p.sa_per_row ? m : 0] : 0.f;
  }
  v4f sbv[WNB][4];
  v2u bv[WNB][4];
#pragma unroll
  for (int j = 0; j < WNB; ++j)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int n = n0 + wn * 32 * WNB + j * 32 + 8 * q + 4 * (lane >> 5);
      sbv[j][q] = v4f{0.f, 0.f, 0.f, 0.f};
      bv[j][q] = v2u{0u, 0u};
      if (n < p.N) {
        if (p.sb_per_col) sbv[j][q] = *reinterpret_cast<const v4f*>(p.sb + n);
        else sbv[j][q] = v4f{p.sb[0], p.sb[0], p.sb[0], p.sb[0]};
        if (p.bias) bv[j][q] = *reinterpret_cast<const v2u*>(p.bias + n);
      }
    }
#pragma unroll
  for (int i = 0; i < WMB; ++i) {
#pragma unroll
    for (int j = 0; j < WNB; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        float o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = sam[i] * (sbv[j][q][r] * acc[i][j][4 * q + r]);
        if (p.bias) {
          o[0] += T::to_float((uint16_t)(bv[j][q].x & 0xffffu));
          o[1] += T::to_float((uint16_t)(bv[j][q].x >> 16));
          o[2] += T::to_float((uint16_t)(bv[j][q].y & 0xffffu));
          o[3] += T::to_float((uint16_t)(bv[j][q].y >> 16));
        }
        v2u ov;
        ov.x = (uint32_t)T::from_float(o[0]) | ((uint32_t)T::from_float(o[1]) << 16);
        ov.y = (uint32_t)T::from_float(o[2]) | ((uint32_t)T::from_float(o[3]) << 16);
        *reinterpret_cast<v2u*>(wave_lds + (lane & 31) * PITCH + (j * 32 + 8 * q + 4 * (lane >> 5)) * 2) = ov;
      }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();           // lanes exchange data through LDS; its operations run in program order
#pragma unroll
    for (int it = 0; it < 32 * CPR / 64; ++it) {
      const int idx = it * 64 + lane;
      const int row = idx / CPR, ch = idx % CPR;
      const v4u v = *reinterpret_cast<const v4u*>(wave_lds + row * PITCH + ch * 16);
      const int m = m0 + wm * 32 * WMB + i * 32 + row;
      const int n = n0 + wn * 32 * WNB + ch * 8;
      if (m < p.M && n < p.N) *reinterpret_cast<v4u*>(p.out + (int64_t)m * p.ldc + n) = v;
    }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
  }
}

// The tail of the multi-stage tile kernels: (split K) hand the partial tile over and let one wavefront sum
// (tile_handover.h), then the scaled epilogue.  `sl` = the workgroup's (tile, K part); `lds8` = at least
// NW * 32 * (WNB * 64 + 16) bytes of LDS that every wavefront of the workgroup is done with.
template <bool BF16_OUT, int WMB, int WNB, int NW>
__device__ inline void fp8_tile_tail(const Fp8MMParams& p, v16f (&acc)[WMB][WNB], uint8_t* lds8, const TileSlot& sl,
                                     int wave, int lane, int m0, int n0, int wm, int wn) {
  if (sl.nsplit > 1 && !handover_finish<WMB, WNB, NW>(p.c_tmp, p.counters, acc, sl, wave, lane)) return;

  if (((uintptr_t)p.out & 15) == 0)
    tile_epilogue_lds<BF16_OUT, WMB, WNB>(p, acc, m0, n0, wm, wn, lane, lds8 + wave * (32 * (WNB * 64 + 16)));
  else
    tile_epilogue<BF16_OUT, WMB, WNB>(p, acc, m0, n0, wm, wn, lane);
}

// ----------------------------------------------------------------------------- tile kernel
template <bool BF16_OUT, int WMB, int WNB>
__global__ __launch_bounds__(256) void fp8_mm_tile_kernel(const Fp8MMParams p) {
  constexpr int BM = 64 * WMB, BN = 64 * WNB;
  constexpr int A_CH = BM / 32, B_CH = BN / 32;   // 16-byte chunks per thread per step
  extern __shared__ __attribute__((aligned(16))) uint8_t lds8[];
  uint8_t* As = lds8;                         // [2][BM][PITCH]
  uint8_t* Bs = lds8 + 2 * BM * F8_PITCH;     // [2][BN][PITCH]

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  const int tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N + BN - 1) / BN;
  const int total = tiles_m * tiles_n;
  int bid = blockIdx.x;
  if (total % 8 == 0) bid = (bid & 7) * (total / 8) + (bid >> 3);   // one contiguous band of tiles per XCD
  const int tm = bid % tiles_m, tn = bid / tiles_m;
  const int m0 = tm * BM, n0 = tn * BN;

  v4u areg[A_CH], breg[B_CH];
  auto load_g = [&](int step) {
    const int kb = step * F8_BK;
#pragma unroll
    for (int i = 0; i < A_CH; ++i) {
      const int c = tid + 256 * i;
      const int row = c >> 3, ch = c & 7;
      const int m = m0 + row, k = kb + ch * 16;
      v4u v = {0u, 0u, 0u, 0u};
      if (m < p.M && k < p.K) v = *reinterpret_cast<const v4u*>(p.a + (int64_t)m * p.lda + k);
      areg[i] = v;
    }
#pragma unroll
    for (int i = 0; i < B_CH; ++i) {
      const int c = tid + 256 * i;
      const int row = c >> 3, ch = c & 7;
      const int n = n0 + row, k = kb + ch * 16;
      v4u v = {0u, 0u, 0u, 0u};
      if (n < p.N && k < p.K) v = *reinterpret_cast<const v4u*>(p.b + (int64_t)n * p.ldb + k);
      breg[i] = v;
    }
  };
  auto store_l = [&](int buf) {
#pragma unroll
    for (int i = 0; i < A_CH; ++i) {
      const int c = tid + 256 * i;
      *reinterpret_cast<v4u*>(As + ((size_t)buf * BM + (c >> 3)) * F8_PITCH + (c & 7) * 16) = areg[i];
    }
#pragma unroll
    for (int i = 0; i < B_CH; ++i) {
      const int c = tid + 256 * i;
      *reinterpret_cast<v4u*>(Bs + ((size_t)buf * BN + (c >> 3)) * F8_PITCH + (c & 7) * 16) = breg[i];
    }
  };

  v16f acc[WMB][WNB];
#pragma unroll
  for (int i = 0; i < WMB; ++i)
#pragma unroll
    for (int j = 0; j < WNB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  const int steps = (p.K + F8_BK - 1) / F8_BK;
  load_g(0);
  store_l(0);
  if (steps > 1) load_g(1);
  __syncthreads();

  for (int step = 0; step < steps; ++step) {
    const int cur = step & 1;
    if (step + 1 < steps) {
      store_l(cur ^ 1);
      if (step + 2 < steps) load_g(step + 2);
    }
    const uint8_t* Ab = As + ((size_t)cur * BM + wm * 32 * WMB + (lane & 31)) * F8_PITCH + (lane >> 5) * 32;
    const uint8_t* Bb = Bs + ((size_t)cur * BN + wn * 32 * WNB + (lane & 31)) * F8_PITCH + (lane >> 5) * 32;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      v8i af[WMB], bf[WNB];
#pragma unroll
      for (int i = 0; i < WMB; ++i) {
        const v4i lo = *reinterpret_cast<const v4i*>(Ab + (size_t)i * 32 * F8_PITCH + kk * 64);
        const v4i hi = *reinterpret_cast<const v4i*>(Ab + (size_t)i * 32 * F8_PITCH + kk * 64 + 16);
        af[i] = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      }
#pragma unroll
      for (int j = 0; j < WNB; ++j) {
        const v4i lo = *reinterpret_cast<const v4i*>(Bb + (size_t)j * 32 * F8_PITCH + kk * 64);
        const v4i hi = *reinterpret_cast<const v4i*>(Bb + (size_t)j * 32 * F8_PITCH + kk * 64 + 16);
        bf[j] = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      }
#pragma unroll
      for (int i = 0; i < WMB; ++i)
#pragma unroll
        for (int j = 0; j < WNB; ++j) acc[i][j] = mfma_fp8_32(bf[j], af[i], acc[i][j]);   // rows = n, columns = m
    }
    __syncthreads();
  }

  tile_epilogue<BF16_OUT, WMB, WNB>(p, acc, m0, n0, wm, wn, lane);
}

// ----------------------------------------------------------------------------- tile kernel, direct-to-LDS variant
// Same tiling as fp8_mm_tile_kernel, but both operand tiles go global -> LDS with `buffer_load_dwordx4 ... lds`
// (no registers, no VALU, no ds_write): each wavefront instruction moves 8 rows x 128 bytes.  The LDS tile is
// unpadded [row][8 chunks of 16 B] with the chunk index XOR-ed by (row & 7), applied on the *global* side (the LDS
// side of such a load is fixed: lane L writes bytes 16L..16L+15), which keeps the 16-byte operand reads of 8
// consecutive rows on 8 different bank groups.  Rows beyond M / N fall outside the buffer descriptor and read as zero.
// Requires K % 128 == 0 (a partial last step would read the neighbouring row instead of zeros).
template <bool BF16_OUT, int WMB, int WNB>
__global__ __launch_bounds__(256) void fp8_mm_tile2_kernel(const Fp8MMParams p) {
  constexpr int BM = 64 * WMB, BN = 64 * WNB;
  constexpr int STAGE = (BM + BN) * 128;          // bytes per stage
  extern __shared__ __attribute__((aligned(16))) uint8_t lds8[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;

  const int tiles_m = (p.M + BM - 1) / BM, tiles_n = (p.N + BN - 1) / BN;
  const int total = tiles_m * tiles_n;
  int bid = blockIdx.x;
  if (total % 8 == 0) bid = (bid & 7) * (total / 8) + (bid >> 3);   // one contiguous band of tiles per XCD
  const int tm = bid % tiles_m, tn = bid / tiles_m;
  const int m0 = tm * BM, n0 = tn * BN;

  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.a), 0, (int)p.a_extent, 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.b), 0, (int)p.b_extent, 0x00020000);
  const int lrow = lane >> 3, lchunk = (lane & 7) ^ lrow;
  const uint32_t voff_a = (uint32_t)lrow * (uint32_t)p.lda + (uint32_t)lchunk * 16u;
  const uint32_t voff_b = (uint32_t)lrow * (uint32_t)p.ldb + (uint32_t)lchunk * 16u;

  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  auto issue_loads = [&](int step, int buf) {
    uint8_t* Ab = lds8 + (size_t)buf * STAGE;
    uint8_t* Bb = Ab + BM * 128;
#pragma unroll
    for (int i = 0; i < BM / 32; ++i) {
      const int r0 = wave * (BM / 4) + i * 8;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(Ab + r0 * 128), 16, (int)voff_a,
                                               (int)((uint32_t)min(m0 + r0, p.M - 1) * (uint32_t)p.lda + (uint32_t)step * 128u), 0, 0);      // (vaq_common.h)
    }
#pragma unroll
    for (int i = 0; i < BN / 32; ++i) {
      const int r0 = wave * (BN / 4) + i * 8;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_ptr_t)(Bb + r0 * 128), 16, (int)voff_b,
                                               (int)((uint32_t)min(n0 + r0, p.N - 1) * (uint32_t)p.ldb + (uint32_t)step * 128u), 0, 0);
    }
  };

  v16f acc[WMB][WNB];
#pragma unroll
  for (int i = 0; i < WMB; ++i)
#pragma unroll
    for (int j = 0; j < WNB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // operand read offsets: row r = lane&31 of a 32-row block, 32 bytes = chunks (kk*4 + kh*2, +1), swizzled by (r & 7)
  const int r7 = lane & 7, kh = lane >> 5;
  uint32_t coff[2][2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk)
#pragma unroll
    for (int h = 0; h < 2; ++h) coff[kk][h] = (uint32_t)(((kk * 4 + kh * 2 + h) ^ r7) * 16);
  const uint32_t arow = (uint32_t)((wm * 32 * WMB + (lane & 31)) * 128);
  const uint32_t brow = (uint32_t)(BM * 128 + (wn * 32 * WNB + (lane & 31)) * 128);

  const int steps = p.K / F8_BK;
  issue_loads(0, 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();

  for (int step = 0; step < steps; ++step) {
    const int cur = step & 1;
    if (step + 1 < steps) issue_loads(step + 1, cur ^ 1);
    const uint8_t* base = lds8 + (size_t)cur * STAGE;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      v8i af[WMB], bf[WNB];
#pragma unroll
      for (int i = 0; i < WMB; ++i) {
        const v4i lo = *reinterpret_cast<const v4i*>(base + arow + i * 4096 + coff[kk][0]);
        const v4i hi = *reinterpret_cast<const v4i*>(base + arow + i * 4096 + coff[kk][1]);
        af[i] = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      }
#pragma unroll
      for (int j = 0; j < WNB; ++j) {
        const v4i lo = *reinterpret_cast<const v4i*>(base + brow + j * 4096 + coff[kk][0]);
        const v4i hi = *reinterpret_cast<const v4i*>(base + brow + j * 4096 + coff[kk][1]);
        bf[j] = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      }
#pragma unroll
      for (int i = 0; i < WMB; ++i)
#pragma unroll
        for (int j = 0; j < WNB; ++j) acc[i][j] = mfma_fp8_32(bf[j], af[i], acc[i][j]);   // rows = n, columns = m
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // next stage has landed in LDS
    __syncthreads();
  }

  tile_epilogue<BF16_OUT, WMB, WNB>(p, acc, m0, n0, wm, wn, lane);
}

// ----------------------------------------------------------------------------- tile kernel, multi-stage direct-to-LDS
// The kernel the M > 32 path normally uses.  Differences from fp8_mm_tile2_kernel:
//  * one MFMA k-slice (64 bytes of K) per stage, NST stages in a ring: the requests for step s+NST-1 go out in
//    step s, so a tile has NST-2 full steps to arrive before anybody waits for it (with two stages of 128
//    bytes the wait at the end of every step saw most of the L2 latency);
//  * vector-memory operations retire in issue order, so "the tile of step s+1 has landed" is `vmcnt <= requests issued
//    after it`, a compile-time constant; the workgroup barrier is the bare instruction (a __syncthreads() carries a fence
//    that drains every outstanding load);
//  * LDS rows are 64 bytes; four rows form one 256-byte line of 16 chunks (chunk index (row & 3) * 4 + c) and the chunk
//    index is XOR-ed with (row >> 2) & 3; or (LINE) 128 bytes, two to a line, the chunk index XOR-ed with bits 1, 3, 2 of the row.  The LDS has 64
//    banks (256 bytes per cycle): 16 lanes reading 16 consecutive rows at the same k chunk touch 16 different 16-byte bank groups;
//  * two slices of K are requested at a time (KS = 2, or PP = 2 where the ring has no room for whole pairs), for the reason at
//    `load` below, and by eight wavefronts even for a 128 x 128 tile: with four a compute unit has fewer requests under
//    way.  128 x 128 tiles, cold: 4096 x 6144 at M = 333 23.3 -> 19.5 us, 5120 x 13824 at M = 250 29.3 -> 24.3 us (cached);
//    256 x 128: 4096 x 4096 at M = 2048 40.7 -> 35.8 us; 256 x 256: 4096 x 4096 at M = 4096 59.0 -> 56.1 us (2.45 PFLOP/s),
//    14336 x 4096 195.5 -> 183.1 us.  Not kept: four slices at a time in two stages, K slices dealt to two groups of
//    wavefronts of the same tile (fewer fragment reads, same time), sixteen wavefronts, four-slice stages of 64 x 64 tiles;
//  * WAVES_M x WAVES_N wavefronts; tiles are handed out in bands of 4 tile rows inside each XCD's contiguous range so
//    that the tiles resident on one XCD share activation rows and weight columns in its L2.
// Requires M*lda, N*ldb < 2^32, and K % 64 == 0, or a multiple of 16 with TAIL: a step that ends past K would read the neighbouring row instead of
// zeros, so that every chunk of 16 bytes is tested and those past K are requested behind the operand's end (8 vector instructions a step; all
// offsets below 2 GiB, see dispatch_tile).
template <bool BF16_OUT, int BM, int BN, int WAVES_M, int WAVES_N, int NST, int KS = 1, int PP = 0, bool TAIL = false>
__global__ __launch_bounds__(WAVES_M * WAVES_N * 64) void fp8_mm_tile3_kernel(VAQ_HEAD_ARGS, const Fp8MMParams p) {
  // what the first requests need (vaq_common.h; see launch_tile3)
  const uint8_t* const a = head_ptr<uint8_t>(h0[0], h0[1]);
  const uint8_t* const b = head_ptr<uint8_t>(h0[2], h0[3]);
  const uint32_t lda = h0[4], ldb = h0[5], tiles_m = h1[2], tiles_n = h1[1], flags = h2[1];      // (rotate_k from bit 16 on)
  const int M = (int)h0[6], N = (int)h0[7], K = (int)h1[0];
  // A step is KS k-slices of 64 bytes (KS = 2 for the small tiles, whose steps are otherwise shorter than the barrier
  // and the LDS round trip that every step pays); a stage holds the KS slices of one step, each as [A tile | B tile].
  constexpr bool PAIR = PP == 2, LINE = KS == 2 || PAIR;        // requests of whole 128-byte lines (see `load`)
  constexpr int NW = WAVES_M * WAVES_N;
  constexpr int TM = BM / WAVES_M, TN = BN / WAVES_N;
  constexpr int WMB = TM / 32, WNB = TN / 32;
  constexpr int A_ST = BM * 64, B_ST = BN * 64, SLICE = A_ST + B_ST, STAGE = KS * SLICE;
  constexpr int A_LD = BM / (16 * NW), B_LD = BN / (16 * NW);     // DMA instructions per wavefront and slice (16 rows each)
  constexpr int LPW = KS * (A_LD + B_LD);
  static_assert(A_LD >= 1 && B_LD >= 1, "tile too small for this many wavefronts");
  static_assert((NST - 2) * LPW <= 63, "wait counter range");
  extern __shared__ __attribute__((aligned(16))) uint8_t lds8[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WAVES_N, wn = wave % WAVES_N;

  const TileSlot sl = tile_slot(TileGrid{tiles_n, tiles_m, h1[3], h2[0], flags}, p);          // one contiguous range of tile positions per XCD
  const int tm = sl.tm, tn = sl.tn;
  const int m0 = tm * BM, n0 = tn * BN;

  // (ends as p.a_extent and p.b_extent, formed here from what comes with the launch)
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a), 0, (int)((uint32_t)(M - 1) * lda + (uint32_t)K), 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(b), 0, (int)((uint32_t)(N - 1) * ldb + (uint32_t)K), 0x00020000);
  // DMA instruction.  One slice: 16 rows x 64 bytes = four 256-byte lines; lane l lands in slot l: line j = r0/4 + (l >> 4), swizzled
  // chunk l & 15 -> c16 = (l & 15) ^ (j & 3), row = 4j + (c16 >> 2), chunk = c16 & 3.  r0 is a multiple of 16, so j & 3 = l >> 4.
  // Two slices (LINE): 8 rows x 128 bytes; row r0 + (l >> 3), chunk (l & 7) ^ f, f = bits 3, 1, 2 of the row in this order -> with r0 = 8 times the
  // instruction's number, bits 5 and 4 of l in places 2 and 0, and 2 more for the odd instructions of a wavefront.
  const int c16 = (lane & 15) ^ (lane >> 4);
  const uint32_t lrow = (uint32_t)(LINE ? lane >> 3 : 4 * (lane >> 4) + (c16 >> 2));
  const uint32_t lbyte = (uint32_t)(LINE ? (lane & 7) ^ ((lane >> 4 & 1) | (lane >> 5) << 2) : c16 & 3) * 16u;
  const uint32_t row_a = lrow * lda, row_b = lrow * ldb;
  const uint32_t voff_a = row_a + lbyte, voff_b = row_b + lbyte;
  const uint32_t voff_a1 = row_a + (lbyte ^ 32u), voff_b1 = row_b + (lbyte ^ 32u);      // (LINE: odd instructions)

  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  // K may be split over workgroups: this one covers the steps [s_lo, s_hi)
  const int all_steps = TAIL ? (K + 64 * KS - 1) / (64 * KS) : K / (64 * KS);
  // (in pairs: parts start at even steps, so that the two slices of a request share their cache lines)
  const auto part = [&](int i) { return i >= sl.nsplit ? all_steps : tile_part(p, sl, all_steps, i) & (PAIR ? ~1 : ~0); };
  const int s_lo = part(sl.split), s_hi = part(sl.split + 1);
  const int steps = s_hi - s_lo;
  // Few tile rows (M at most 4 tiles high) on a device that the tiles do not fill: the tiles of one column would read
  // the same weight rows at the same time, which leaves only (ring depth x 64 KS) bytes per weight row in flight --
  // with cold weights the kernel then runs at a fraction of the memory bandwidth.  Tile row tm starts its K loop
  // tm / tiles_m of the way into its range and wraps around: the rows are read at tiles_m places at once, and the later
  // readers find them in the L2 (4096 x 4096 at M = 256, cold: 24.4 -> 18.3 us).
  // rotate_k = 2, one or two tile rows on a wide layer: every workgroup reads the same activation rows, and with K a power
  // of two all of them ask the same few L2 channels for the same lines at the same time.  Tile column tn starts tn / tiles_n
  // of the way into K instead (4096 x 28672 at M = 72 .. 256, cold: 33.9 .. 45.4 -> 31.1 .. 43.6 us; no change on K = 3584 or
  // 5120; with 16 tile rows it costs 3-9 %: the tiles of one column then no longer read their weights together).
  int rot = 0;
  if (const uint32_t rotate_k = flags >> 16; rotate_k != 0)
    rot = (int)div_by((uint32_t)((rotate_k == 1 ? tm : tn) * steps), rotate_k == 1 ? tiles_m : tiles_n, p.rotate_magic);
  if (PAIR) rot = steps & 1 ? 0 : rot & ~1;      // a pair never wraps around
  // Requests for ROWS rows of an operand, from row `first` and K byte `koff` on.  LINE: eight lanes ask for 128 bytes, a whole cache line,
  // which crosses from the L2 in one piece; else the slices of a step row by row, whose halves of a line cross one after the other.  Weights from
  // memory, halves -> lines: 128 x 128 tiles: 5120 x 13824 at M = 250 33.6 -> 31.5 us, 4096 x 28672 at M = 100 30.3 -> 27.7; 64 x 128, 128 x 64, 128 x 256:
  // 2 - 9 %; 64 x 64: 3 - 6 %; 256 x 256: 4096 x 28672 at M = 512 59.1 -> 56.1; from the memory-side cache level.  Pieces of 256 bytes (four slices,
  // half of the rows at a time): -4 .. +3 % against lines; one operand in lines and the other in halves: in between.
  // Rows from `last` + 1 on are not there (vaq_common.h): of those that begin at one of them, the first eighth (quarter) of the lanes gets the last row, the others zeros.
  auto load = [&](auto rows, const __amdgpu_buffer_rsrc_t& r, uint32_t first, uint32_t last, uint32_t pitch, uint32_t v0, uint32_t v1, uint32_t koff, uint8_t* at) {
    constexpr int ROWS = decltype(rows)::value;
    if constexpr (LINE) {
      constexpr int LD = ROWS / (8 * NW);
#pragma unroll
      for (int i = 0; i < LD; ++i) {
        const int r0 = (wave * LD + i) * 8;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)(at + r0 * 128), 16, (int)(i & 1 ? v1 : v0), (int)(min(first + (uint32_t)r0, last) * pitch + koff), 0, 0);
      }
    } else {
      constexpr int LD = ROWS / (16 * NW);
#pragma unroll
      for (int i = 0; i < LD; ++i) {
        const int r0 = (wave * LD + i) * 16;
#pragma unroll
        for (int c = 0; c < KS; ++c)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)(at + (c * ROWS + r0) * 64), 16, (int)v0, (int)(min(first + (uint32_t)r0, last) * pitch + koff + 64u * c), 0, 0);
      }
    }
  };
  // (a chunk past K: an offset past either operand's end)
  static_assert(!TAIL || LINE, "chunks past K of single slices are not built");
  auto in_k = [&](uint32_t offset, uint32_t byte) { return !TAIL || byte < (uint32_t)K ? offset : 0x80000000u; };
  auto load_a = [&](uint32_t koff, uint8_t* at) {
    load(std::integral_constant<int, BM>{}, ra, (uint32_t)m0, (uint32_t)M - 1u, lda, in_k(voff_a, koff + lbyte), in_k(voff_a1, koff + (lbyte ^ 32u)), koff, at);
  };
  auto load_b = [&](uint32_t koff, uint8_t* at) {
    load(std::integral_constant<int, BN>{}, rb, (uint32_t)n0, (uint32_t)N - 1u, ldb, in_k(voff_b, koff + lbyte), in_k(voff_b1, koff + (lbyte ^ 32u)), koff, at);
  };
  // Steps are requested in order: the first byte of K of the next one, rotation applied.  (As few scalar instructions as can be: the matrix
  // cores wait for them at the start of every step.)
  constexpr uint32_t K_STEP = PAIR ? 128 : 64 * KS;
  const uint32_t k_lo = (uint32_t)s_lo * 64u * KS, k_hi = (uint32_t)s_hi * 64u * KS;
  uint32_t k_at = k_lo + (uint32_t)rot * 64u * KS;
  auto next_k = [&] {
    const uint32_t k = k_at;
    k_at = k + K_STEP >= k_hi ? k_lo : k + K_STEP;
    return k;
  };
  auto request = [&](int stage) {
    uint8_t* const at = lds8 + (size_t)stage * STAGE;
    const uint32_t k = next_k();
    load_a(k, at);
    load_b(k, at + KS * A_ST);
  };

  v16f acc[WMB][WNB];
#pragma unroll
  for (int i = 0; i < WMB; ++i)
#pragma unroll
    for (int j = 0; j < WNB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // operand reads: row = lane & 31 of a 32-row block (blocks start at multiples of 32 rows), the lane's 32 bytes are
  // chunks 2*kh and 2*kh+1 (kh = lane >> 5) of the slice.  The 16 lanes that are served together read 16 rows at the same chunk of K: 16
  // different places of a 256-byte line in either layout.
  const int kh = lane >> 5;
  uint32_t coff[2];
#pragma unroll
  for (int h = 0; h < 2; ++h)
    coff[h] = LINE ? (uint32_t)((lane & 31) * 128 + (((kh * 2 + h) ^ ((lane >> 1 & 1) | (lane >> 2 & 1) << 2 | (lane >> 3 & 1) << 1)) * 16))
                   : (uint32_t)(((lane & 31) >> 2) * 256 + ((((lane & 3) * 4 + kh * 2 + h) ^ ((lane >> 2) & 3)) * 16));
  // LDS addresses of this wavefront's fragments at the step at hand, slice ks (LINE: half ks of each line)
  typedef __attribute__((address_space(3))) const v4i* lds_v4i_t;
  constexpr int SL = LINE ? 2 : 1, ROW_BYTES = LINE ? 128 : 64, PLACE = (BM > BN ? BM : BN) * 128;      // (PLACE: see PP = 2)
  uint32_t adr_a[SL][2], adr_b[SL][2];
  {
    const uint32_t base = (uint32_t)(uintptr_t)(lds_ptr_t)lds8;
#pragma unroll
    for (int ks = 0; ks < SL; ++ks)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t at = base + (coff[h] ^ (ks ? 64u : 0u));
        adr_a[ks][h] = at + (uint32_t)(wm * TM * ROW_BYTES + (PAIR ? PLACE : 0));
        adr_b[ks][h] = at + (uint32_t)(wn * TN * ROW_BYTES + (PAIR ? 0 : KS * A_ST));
      }
  }
  auto fragment = [&](const uint32_t (&adr)[2], int block) {
    const v4i lo = *reinterpret_cast<lds_v4i_t>((uintptr_t)(adr[0] + block * 32 * ROW_BYTES));
    const v4i hi = *reinterpret_cast<lds_v4i_t>((uintptr_t)(adr[1] + block * 32 * ROW_BYTES));
    return v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
  };
  auto read_a = [&](int ks, v8i (&af)[WMB]) {
#pragma unroll
    for (int i = 0; i < WMB; ++i) af[i] = fragment(adr_a[ks], i);
  };
  auto read_b = [&](int ks, v8i (&bf)[WNB]) {
#pragma unroll
    for (int j = 0; j < WNB; ++j) bf[j] = fragment(adr_b[ks], j);
  };
  // (here and now, in the shadow of the reads: the compiler would rather add ahead of the next reads, with everybody waiting)
  auto move = [&](uint32_t (&adr)[SL][2], int by) {
#pragma unroll
    for (int ks = 0; ks < SL; ++ks)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        adr[ks][h] += (uint32_t)by;
#ifdef __HIP_DEVICE_COMPILE__
        asm volatile("" : "+v"(adr[ks][h]));
#endif
      }
  };

  // (Reading the fragments of step s+1 during the MFMAs of step s -- one more stage of slack, double-buffered weight
  // fragments -- was measured 5% slower than reading them at the start of their own step, and is not done.)
  //
  // A step is a chain -- barrier, addresses, fragment reads, MFMAs -- that every wavefront of the workgroup walks through together, so that what
  // stands ahead of the reads is paid in full.  The addresses are held, and moved on (`by` bytes) behind the reads; the reads come first, of both slices
  // where the registers hold them (at most two blocks to a wavefront), the requests behind them; the loops stay rolled.  With whole lines, drawn problems,
  // weights from the memory-side cache / from memory, against addresses computed ahead of the reads and requests of halves ahead of them: 128 x 128
  // tiles -4 / -5 % (5120 x 13824 at M = 250 26.0 -> 24.7 us with its quantisation), 64 x 128 -5 / -7, 128 x 64 -6 / -6, 64 x 64 -3 / -3, 128 x 256 -3 / -3, 256 x 128
  // -10 / -9, 256 x 256 -5 / -5 (14336 x 4096 at M = 4096 183 -> 163 us, 4096 x 28672 at M = 2048 218 -> 200).  Written out for a turn of the ring, with the stages in
  // the reads' offsets, a long K gains up to 5 % more, but a short one waits for the larger code: 2944 x 8896 at M = 1759 47 -> 51 us, 1152 x 28288 at
  // M = 492 25.2 -> 27.6.
  constexpr bool AT_ONCE = KS == 1 || WMB * WNB <= 2;
  auto compute = [&](int by, auto requests) {
    if constexpr (AT_ONCE) {
      v8i af[KS][WMB], bf[KS][WNB];
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        read_b(ks, bf[ks]);
        read_a(ks, af[ks]);
      }
      if constexpr (PP == 0) {      // (256 x 384 has no registers for all of them at once)
        __builtin_amdgcn_sched_barrier(0);
        requests();
        move(adr_a, by);
        move(adr_b, by);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int i = 0; i < WMB; ++i)
#pragma unroll
          for (int j = 0; j < WNB; ++j) acc[i][j] = mfma_fp8_32(bf[ks][j], af[ks][i], acc[i][j]);   // rows = n, columns = m
    } else {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        v8i af[WMB], bf[WNB];
        read_b(ks, bf);
        read_a(ks, af);
        __builtin_amdgcn_sched_barrier(0);
        if (ks == 0) requests();
        if (ks == KS - 1) {
          move(adr_a, by);
          move(adr_b, by);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < WMB; ++i)
#pragma unroll
          for (int j = 0; j < WNB; ++j) acc[i][j] = mfma_fp8_32(bf[j], af[i], acc[i][j]);
      }
    }
  };
  auto nothing = [] {};
  // end of a step: LDS reads of this wavefront done, requests older than the newest `n` landed, then the bare barrier
  auto sync_step = [&](auto n_c) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(decltype(n_c)::value) : "memory");
  };
  using WAIT_STEADY = std::integral_constant<int, (NST - 2) * LPW>;
  using WAIT_NONE = std::integral_constant<int, 0>;

  // Invariant at the start of step s: the tile of step s complete in LDS, the tiles of steps s+1 .. s+NST-2 requested,
  // stage (s-1) % NST free.  The requests of step s+NST-1 go out in step s, behind its first fragment reads.
  // Alternating phases (PP): the two wavefronts that share a SIMD run half a step apart, so that one reads its fragments
  // (and requests operands) while the other one issues its MFMAs.  A step is [requests, fragment reads, wait] barrier
  // [MFMAs] barrier; the late half of the workgroup passes one extra barrier first and skips its last one, so every
  // wavefront passes the same number.  What the next step reads must have landed at the END OF THE READ PHASE of this one
  // (the early half reads it two barriers later, the late half three).
  auto mfmas = [&](v8i (&af)[WMB], v8i (&bf)[WNB]) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < WMB; ++i)
#pragma unroll
      for (int j = 0; j < WNB; ++j) acc[i][j] = mfma_fp8_32(bf[j], af[i], acc[i][j]);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto bare_barrier = [&]() { asm volatile("s_barrier" ::: "memory"); };
  const bool late = wave >= NW / 2;     // wavefronts w and w + 4 share a SIMD (the other pairing measured 10-25 % slower)
  if constexpr (PAIR) {
    // Two steps read the two slices of a pair of them, 128 bytes of every row, the weights of both in the first.  The LDS has five places for
    // an operand of a pair, which weights and activations take in turn, B(0) A(0) B(1) A(1) ...: those of the pair at hand, of the next, and
    // the weights of the one after that.  The weights are free after a pair's first step, the activations after its second, and each
    // is at once replaced by what comes two and a half pairs later, so that a request has three or four steps to be answered.
    // (Both operands free after the second step: two and four steps, 4 % slower on 4096 x 28672 at M = 4096.)  A step is bound by its chain of
    // reads and MFMAs and by the power limit: with all operands zero 4096^3 takes 0.7 of the time, without any MFMA half.
    static_assert(BM == BN && NST == 5, "five places of one size");
    constexpr int LD = BM / (8 * NW);                          // requests of a wavefront for an operand of a pair
    const int pairs = (steps + 1) / 2;                         // (the last one may be half a pair: what follows it is requested, up to the end of the operand, and not read)
    int qb = 0;                                                // place of the pair at hand's weights
    auto place = [&](int ahead) {                              // that of the operand `ahead` places on
      const int q = qb + ahead;
      return lds8 + (q >= 5 ? q - 5 : q) * PLACE;
    };
    {
      const uint32_t k0 = next_k(), k1 = next_k();
      load_b(k0, place(0));
      load_a(k0, place(1));
      if (pairs > 1) {
        load_b(k1, place(2));
        load_a(k1, place(3));
        sync_step(std::integral_constant<int, 2 * LD>{});      // the first pair landed
      } else {
        sync_step(WAIT_NONE{});
      }
    }
    if (late) bare_barrier();
    v8i af[WMB], bf[2][WNB];
    auto places_on = [](int q) { return q >= 3 ? -3 * PLACE : 2 * PLACE; };      // from place q to the next pair's
    int pair = 0;
#pragma unroll 1
    for (; pair < steps / 2; ++pair) {
      const bool more = pair + 2 < pairs;
      const uint32_t k = next_k();
      read_a(0, af);
      read_b(0, bf[0]);
      read_b(1, bf[1]);
      __builtin_amdgcn_sched_barrier(0);
      if (more) load_b(k, place(4));
      move(adr_b, places_on(qb));
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      mfmas(af, bf[0]);
      bare_barrier();
      read_a(1, af);
      __builtin_amdgcn_sched_barrier(0);
      if (more) load_a(k, place(0));
      move(adr_a, places_on(qb == 4 ? 0 : qb + 1));
      if (more) sync_step(std::integral_constant<int, 2 * LD>{});      // the next pair landed
      else sync_step(WAIT_NONE{});
      mfmas(af, bf[1]);
      if (!late || 2 * pair + 2 < steps) bare_barrier();
      qb = qb >= 3 ? qb - 3 : qb + 2;
    }
    if (steps & 1) {      // half a pair
      read_a(0, af);
      read_b(0, bf[0]);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      mfmas(af, bf[0]);
      if (!late) bare_barrier();
    }
  } else if (PP == 1 && steps >= NST) {
    // (256 x 384: the registers are full, so that stages and requests are computed step by step)
    auto k_of = [&](int step) {
      const int rel = step - s_lo + rot;
      return (uint32_t)(s_lo + (rel >= steps ? rel - steps : rel)) * 64u;
    };
    auto issue_loads = [&](int step, int stage) {
      uint8_t* const at = lds8 + (size_t)stage * STAGE;
      load_a(k_of(step), at);
      load_b(k_of(step), at + A_ST);
    };
#pragma unroll
    for (int s0 = 0; s0 < NST - 1; ++s0) issue_loads(s_lo + s0, s0);
    sync_step(WAIT_STEADY{});           // the first tile landed
    if (late) bare_barrier();
    int cur = 0, dst = NST - 1;
    auto next = [](int stage) { return stage + 1 == NST ? 0 : stage + 1; };
    auto at = [&](int stage) { return lds8 + (size_t)stage * STAGE; };
    auto fragments = [&](const uint8_t* rows, auto& f) {
#pragma unroll
      for (int i = 0; i < (int)(sizeof(f) / sizeof(v8i)); ++i) {
        const v4i lo = *reinterpret_cast<const v4i*>(rows + i * 2048 + coff[0]), hi = *reinterpret_cast<const v4i*>(rows + i * 2048 + coff[1]);
        f[i] = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      }
    };
    int step = 0;
    for (; step + NST - 1 < steps; ++step) {
      issue_loads(s_lo + step + NST - 1, dst);
      v8i af[WMB], bf[WNB];
      fragments(at(cur) + A_ST + wn * TN * 64, bf);
      fragments(at(cur) + wm * TM * 64, af);
      sync_step(WAIT_STEADY{});
      mfmas(af, bf);
      bare_barrier();
      cur = next(cur);
      dst = next(dst);
    }
    for (; step < steps; ++step) {      // nothing left to request: drain
      v8i af[WMB], bf[WNB];
      fragments(at(cur) + A_ST + wn * TN * 64, bf);
      fragments(at(cur) + wm * TM * 64, af);
      sync_step(WAIT_NONE{});
      mfmas(af, bf);
      if (!(late && step == steps - 1)) bare_barrier();
      cur = next(cur);
    }
  } else if (steps >= NST) {
#pragma unroll
    for (int s0 = 0; s0 < NST - 1; ++s0) request(s0);
    sync_step(WAIT_STEADY{});           // tile 0 landed
    int cur = 0, dst = NST - 1;
    int step = 0;
    auto next = [](int stage) { return stage + 1 == NST ? 0 : stage + 1; };
#pragma unroll 1
    for (; step + NST - 1 < steps; ++step) {
      compute((next(cur) - cur) * STAGE, [&] { request(dst); });
      sync_step(WAIT_STEADY{});
      cur = next(cur);
      dst = next(dst);
    }
#pragma unroll 1
    for (; step < steps; ++step) {      // nothing left to request: drain
      compute((next(cur) - cur) * STAGE, nothing);
      sync_step(WAIT_NONE{});
      cur = next(cur);
    }
  } else {
    // short K: no ring, one tile at a time
    for (int step = 0; step < steps; ++step) {
      request(0);
      sync_step(WAIT_NONE{});
      compute(0, nothing);
      sync_step(WAIT_NONE{});
    }
  }

  static_assert(NST * STAGE >= NW * 32 * (WNB * 64 + 16), "operand ring too small for the epilogue staging");
  if (m0 >= p.M) return;      // a tile row past M (m_tiles_extra): nothing to hand over or store
  fp8_tile_tail<BF16_OUT, WMB, WNB, NW>(p, acc, lds8, sl, wave, lane, m0, n0, wm, wn);
}

// ----------------------------------------------------------------------------- stream kernel (M <= 32, narrow layers M <= 64)
// blockDim = (64, WK).  Wavefront w owns K steps [w*KS, (w+1)*KS) of 128 bytes; activations of that slab live in
// registers for the whole kernel; the workgroup walks a contiguous range of 16-row weight tiles.
template <bool BF16_OUT, int KS, int MB, bool HALVES = false, bool PF = true>
__global__ __launch_bounds__(512) void fp8_mm_stream_kernel(VAQ_HEAD_ARGS, const Fp8MMParams rest) {
  const Fp8MMParams p = stream_params(h0, h1, h2, rest);
  const int WK = (int)(h1[1] >> 16);
  using T = F16Traits<BF16_OUT>;
  extern __shared__ v4f red[];   // [2][WK][MB][64]
  const int lane = threadIdx.x, w = threadIdx.y;
  const int q = lane >> 4, r16 = lane & 15;
  // HALVES (gridDim.y = 2): the K range is split over two workgroups (the second starts where the slabs of the first
  // end); their partial tiles are summed by whichever arrives last (see the hand-over below).  A template parameter,
  // because the extra live values cost the other instances registers they do not have (14 steps: 12 -> 260 bytes spilled).
  const int kbase = ((HALVES ? (int)blockIdx.y * WK : 0) + w) * KS * 128 + q * 32;

  // Operand loads go through buffer descriptors (the host checks that both operands end below 2 GiB): a 16-byte piece
  // past K or past the last row gets an offset beyond the descriptor's extent and arrives as zeros -- one compare and
  // one select per load instead of a branch and eight zeroed registers.
  constexpr uint32_t OOB = 0x80000000u;
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.a), 0, (int)p.a_extent, 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(p.b), 0, (int)p.b_extent, 0x00020000);
  v8i breg[KS][MB];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
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

  v4i wlo[KS], whi[KS];
  // `live` = false requests nothing (offsets beyond the extent): the request for the tile after the last one stays in
  // the instruction stream, so that the count of loads in flight -- which the waits are derived from -- is the same on
  // every path (behind a branch the compiler assumes the shorter path and waits for the next tile's loads as well).
  auto issue = [&](int nt, int s, bool live) {
    const int k = kbase + s * 128;
    const uint32_t base = (uint32_t)(nt * 16 + r16) * (uint32_t)p.ldb + (uint32_t)k;
    const uint32_t o_lo = (live && k < p.K) ? base : OOB, o_hi = (live && k + 16 < p.K) ? base + 16u : OOB;
    wlo[s] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rb, (int)o_lo, 0, 2));     // 2: streamed once
    whi[s] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(rb, (int)o_hi, 0, 2));
  };
#pragma unroll
  for (int s = 0; s < KS; ++s) issue(nt0, s, nt0 < nt1);
  VAQ_ARRIVED4(p.sb, p.bias, p.out, p.sb_per_col);

  // Epilogue operands are requested ahead of their use (a load issued after the reduction would stall the reducing
  // wavefront, and through the next barrier the whole workgroup, for a memory round trip per n-tile): the activation
  // scales once per kernel, the weight scales and the bias of an n-tile before its MFMAs.  With 14 steps per wavefront
  // there are no registers to spare for that: there they are requested after the tile's last MFMA (14336 x 4096 at
  // M = 1 / 16: 16.5 / 20.8 -> 15.7 / 19.6 us).  Requesting the first tile's weights before the activations was slower
  // on every shape (3-5 %, and 40 % with 14 steps, where it changes what the compiler spills).
  constexpr bool AHEAD = KS < 14;
  const bool reducer_wave = WK > 1 ? w < MB : true;
  float sam_mb[MB];
  if constexpr (AHEAD) {
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const int m = mb * 16 + r16;
      sam_mb[mb] = (reducer_wave && m < p.M) ? p.sa[p.sa_per_row ? m : 0] : 0.f;
    }
  }

  int parity = 0;
  // One n-tile.  PF: request the next tile's weights behind each step's MFMAs.  Launches in which every workgroup has a
  // single tile use the instance without those requests (they would be 2 KS loads that fetch nothing but still pass
  // through the load path: 14336 x 4096 at M = 1 / 16 15.4 / 19.2 -> 16.0 / 20.2 us); as a run-time condition the compiler
  // would derive the waits of the multi-tile case from the shorter path and wait for the next tile's loads too, and
  // both variants in one kernel cost registers (spills with 8 steps and two m-blocks).
  auto do_tile = [&](int nt) {
    v4f acc[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) acc[mb] = v4f{0.f, 0.f, 0.f, 0.f};
    float sb_r[4] = {0.f, 0.f, 0.f, 0.f};
    uint16_t bias_r[4] = {0, 0, 0, 0};
    if constexpr (AHEAD) {
      if (reducer_wave) {
        const int n = nt * 16 + q * 4;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          sb_r[r] = p.sb[p.sb_per_col ? n + r : 0];
          if (p.bias) bias_r[r] = p.bias[n + r];
        }
      }
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const v8i aop = v8i{wlo[s].x, wlo[s].y, wlo[s].z, wlo[s].w, whi[s].x, whi[s].y, whi[s].z, whi[s].w};
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[mb] = mfma_fp8_16(aop, breg[s][mb], acc[mb]);
      // the step's registers are free once its MFMAs have issued: request the next tile's step into them right away
      // (the fence keeps the compiler from collecting these requests behind the tile's last MFMA)
      if constexpr (PF) {
        issue(nt + 1, s, nt + 1 < nt1);
        __builtin_amdgcn_sched_barrier(0);
      }
    }

    if constexpr (!AHEAD) {
      // registers are full until the last MFMA of the tile: request the epilogue operands now, across the reduction
      static_assert(AHEAD || MB == 1, "14 steps per wavefront only with one m-block");
      if (reducer_wave) {
        const int n = nt * 16 + q * 4;
        sam_mb[0] = r16 < p.M ? p.sa[p.sa_per_row ? r16 : 0] : 0.f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          sb_r[r] = p.sb[p.sb_per_col ? n + r : 0];
          if (p.bias) bias_r[r] = p.bias[n + r];
        }
      }
    }

    v4f tot = v4f{0.f, 0.f, 0.f, 0.f};
    bool reducer = w < MB;
    if (WK > 1) {
      v4f* buf = red + (size_t)parity * WK * MB * 64;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) buf[(w * MB + mb) * 64 + lane] = acc[mb];
      __syncthreads();
      if (reducer)
        for (int ww = 0; ww < WK; ++ww) tot += buf[(ww * MB + w) * 64 + lane];
      parity ^= 1;
    } else {
      reducer = true;
    }
    if (HALVES && reducer) {
      // Hand-over as in the tile kernel: the partial tile goes out in device-scope 16-byte stores, one arrival counter
      // per (n-tile, m-block); the workgroup that arrives last adds the parts in the order of the K halves and returns the
      // counter to zero.  (WK > 1 always here: the host splits only a long K.)
      constexpr int SC1 = 16;
      const uint32_t units = (uint32_t)NT * (uint32_t)MB;
      const uint32_t unit = (uint32_t)nt * (uint32_t)MB + (uint32_t)w;
      const __amdgpu_buffer_rsrc_t rt =
          __builtin_amdgcn_make_buffer_rsrc(p.c_tmp, 0, (int)(units * gridDim.y * 1024u), 0x00020000);
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, tot), rt, lane * 16,
                                             (int)((blockIdx.y * units + unit) * 1024u), SC1);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");        // partial tile acknowledged before the counter moves
      int32_t* ctr = p.counters + unit;
      int old = 0;
      if (lane == 0) old = __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      old = __builtin_amdgcn_readfirstlane(old);      // lane 0 holds it; a scalar keeps what depends on it scalar
      if (old != (int)gridDim.y - 1) {
        reducer = false;
      } else {
        v4f sum = {0.f, 0.f, 0.f, 0.f};
        for (uint32_t h = 0; h < gridDim.y; ++h) {
          const v4u r = __builtin_amdgcn_raw_buffer_load_b128(rt, lane * 16, (int)((h * units + unit) * 1024u), SC1);
          sum += __builtin_bit_cast(v4f, r);
        }
        tot = sum;
        if (lane == 0) __hip_atomic_store(ctr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    if (reducer) {
      const int mb_lo = (WK > 1) ? w : 0, mb_hi = (WK > 1) ? w + 1 : MB;
      auto emit = [&](int mb, float sam, const float* sbv, const uint16_t* bsv) {
        const v4f val = (WK > 1) ? tot : acc[mb];
        const int m = mb * 16 + r16;
        if (m < p.M) {
#pragma clang fp contract(off)      // sa * (sb * acc), then + bias: two fp32 roundings, like the tile kernels
          const int n = nt * 16 + q * 4;
          float o[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            o[r] = sam * (sbv[r] * val[r]);
            if (p.bias) o[r] += T::to_float(bsv[r]);
          }
          v2u ov;
          ov.x = (uint32_t)T::from_float(o[0]) | ((uint32_t)T::from_float(o[1]) << 16);
          ov.y = (uint32_t)T::from_float(o[2]) | ((uint32_t)T::from_float(o[3]) << 16);
          *reinterpret_cast<v2u*>(p.out + (int64_t)m * p.ldc + n) = ov;
        }
      };
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)       // unrolled: sam_mb stays in registers
        if (mb >= mb_lo && mb < mb_hi) emit(mb, sam_mb[mb], sb_r, bias_r);
    }
  };
  if constexpr (PF) {
    for (int nt = nt0; nt < nt1; ++nt) do_tile(nt);
  } else {
    if (nt0 < nt1) do_tile(nt0);       // the launcher picks this instance only for one tile per workgroup
  }
}

// ----------------------------------------------------------------------------- host side

// Overrides for tests and benchmarks come through tuning() (all zero = automatic): fp8_path 1 stream / 2 tile,
// fp8_tile_impl 1 = register-staged tile kernel, fp8_tile_cfg = fixed multi-stage tile shape (-1: two-stage kernel),
// fp8_split = K split of the tile kernel, fp8_gx = stream-kernel grid, fp8_stream_split -1 = no two-halves stream route.

template <bool BF16_OUT, int WMB, int WNB>
static int launch_tile(const Fp8MMParams& p, hipStream_t s) {
  constexpr int BM = 64 * WMB, BN = 64 * WNB;
  const size_t lds = (size_t)2 * (BM + BN) * F8_PITCH;
  auto kern = fp8_mm_tile_kernel<BF16_OUT, WMB, WNB>;
  static size_t reserved[VAQ_MAX_DEVICES];
  if (const int rc = reserve_dynamic_lds(reinterpret_cast<const void*>(kern), lds, reserved, "fp8_scaled_mm"); rc != VAQ_OK) return rc;
  const int tiles = ((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
  hipLaunchKernelGGL(kern, dim3(tiles), dim3(256), lds, s, p);
  return VAQ_OK;
}

template <bool BF16_OUT, int WMB, int WNB>
static int launch_tile2(const Fp8MMParams& p, hipStream_t s) {
  constexpr int BM = 64 * WMB, BN = 64 * WNB;
  const size_t lds = (size_t)2 * (BM + BN) * 128;
  auto kern = fp8_mm_tile2_kernel<BF16_OUT, WMB, WNB>;
  static size_t reserved[VAQ_MAX_DEVICES];
  if (const int rc = reserve_dynamic_lds(reinterpret_cast<const void*>(kern), lds, reserved, "fp8_scaled_mm"); rc != VAQ_OK) return rc;
  const int tiles = ((p.M + BM - 1) / BM) * ((p.N + BN - 1) / BN);
  hipLaunchKernelGGL(kern, dim3(tiles), dim3(256), lds, s, p);
  return VAQ_OK;
}

template <bool BF16_OUT, int BM, int BN, int WAVES_M, int WAVES_N, int NST, int KS = 1, int PP = 0, bool TAIL = false>
static int launch_tile3(const Fp8MMParams& p_in, hipStream_t s) {
  Fp8MMParams p = p_in;
  const size_t lds = (size_t)NST * KS * (BM + BN) * 64;
  auto kern = fp8_mm_tile3_kernel<BF16_OUT, BM, BN, WAVES_M, WAVES_N, NST, KS, PP, TAIL>;
  static size_t reserved[VAQ_MAX_DEVICES];
  if (const int rc = reserve_dynamic_lds(reinterpret_cast<const void*>(kern), lds, reserved, "fp8_scaled_mm"); rc != VAQ_OK) return rc;
  const int tiles_m = (p.M + BM - 1) / BM + p.m_tiles_extra, tiles_n = (p.N + BN - 1) / BN, tiles = tiles_m * tiles_n;
  const TileGrid g = tile_grid(tiles_m, tiles_n, p.SK, p.tail_first);
  p.split_magic = tile_split_magic(tiles, p.SK, p.tail_first);
  p.rotate_magic = div_magic((uint32_t)(p.rotate_k == 1 ? tiles_m : tiles_n));
  const dim3 grid = p.tail_first > 0 ? dim3(p.tail_first + (tiles - p.tail_first) * p.SK) : dim3(tiles, p.SK);
  hipLaunchKernelGGL(kern, grid, dim3(WAVES_M * WAVES_N * 64), lds, s,
                     (v8u{ptr_lo(p.a), ptr_hi(p.a), ptr_lo(p.b), ptr_hi(p.b), (uint32_t)p.lda, (uint32_t)p.ldb, (uint32_t)p.M, (uint32_t)p.N}),
                     (v4u{(uint32_t)p.K, g.n, g.m, g.band_magic}), (v2u{g.per8, g.flags | (uint32_t)p.rotate_k << 16}), p);
  return VAQ_OK;
}

// The tile shapes of the multi-stage kernel (ids above 10 take two slices of K a step; asked for, id - 10 is the same).
// Fitted to 2064 problems with M = 9 .. 8192, half of them with K = 1024 .. 14336 and N = 1024 .. 28672, half with K = 256 .. 28672 and
// N = 256 .. 152064, drawn over the logarithm, every shape and K split of each timed on cold weights (30154 launches,
// the first half of those in profiles/plan_prices).  Over all 5493 problems there (91351 launches) the plan with the least predicted
// time is on average 0.8 % slower than the fastest (99 of 100 less than 15 %), where rules by size were 11 % slower at M = 33 .. 1024 (4096 x 13824 at M = 384 49 -> 33 us,
// 8192 x 4096 at M = 180 25 -> 19 us, 14336 x 2048 at M = 384 39 -> 27 us).  Constants fitted to the first half's sizes alone lost 4.3 % at
// N > 28672 and 3.5 % at K or N below 1024 (5120 x 152064 at M = 384 400 -> 326 us, 896 x 4864 at M = 2048 24.2 -> 18.8 us with these).
// (Timed when every shape still requested halves of lines.  4595 problems timed again with whole lines: 1.0 % with these constants, 0.8 % with new
// ones, which over layers that stay in the memory-side cache choose worse by as much, up to 20 % where the two best plans change places.)
constexpr TileShape FP8_TILE_SHAPES[] = {
    {13, 128, 128, 8, 1, 3.48, 0.205, 0.0739, 0, 0}, {14, 64, 128, 4, 1, 3.05, 0.161, 0.118, 0, 0},
    {15, 64, 64, 4, 2, 1.63, 0.103, 0.0209, 0.173, 0}, {16, 128, 64, 4, 1, 2.69, 0.158, 0.0327, 0, 0},
    {17, 128, 256, 8, 1, 5.22, 0.354, 0.17, 0, 0}, {19, 256, 128, 8, 1, 4.93, 0.32, 0.107, 0, 0},
    {1, 256, 256, 8, 1, 7.24, 0.524, 0.118, 0, 0}, {10, 256, 384, 8, 1, 18.4, 0.594, 0.38, 0, 0}};
// The hand-over is priced 1 us above its fit (1.14): a call under graph capture fills counters of its own ahead of a split K, 2.3 us
// a replay.  Mean over the problems, plans chosen with 1.14 / 2.14 / 3.44 against the fastest: 0.5 / 0.7 / 1.2 % slower without
// that fill, 0.7 / 0.5 / 0.4 % with it (9 .. 256 rows 0.6 / 0.9 / 1.7 and 1.0 / 0.5 / 0.4 %); 4096 x 6144 at M = 40 .. 64 stays
// whole: 11.3 .. 12.0 -> 11.1 us; as the operator's call replayed from a graph 14.4 -> 11.9 us at M = 64, 4096 x 4096 13.0 -> 10.8.
// (The last constant, by hand: 1.0 against none, 1.3 against 0.9 % in the mean over the problems whose plan has an odd number of parts.)
constexpr TileCosts FP8_TILE_COSTS = {0.149, 2.14, 0.56, 0.254, 1.0};

static TilePlan make_plan_tile3(int M, int N, int K) {
  const int64_t cus = num_cus_current_device();
  const int steps = (K + 63) / 64;
  const VaqTuning& tn = tuning();
  TilePlan best;
  for (const TileShape& t : FP8_TILE_SHAPES) {
    if (tn.fp8_tile_cfg > 0 ? tn.fp8_tile_cfg != t.id && tn.fp8_tile_cfg != t.id - 10 : t.id == 10 && N % 384 != 0) continue;
    if (K % 64 != 0 && t.id == 10) continue;      // (no registers for the test of chunks past K)
    const int64_t tiles = (int64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn);
    const int64_t rest = tiles % cus;
    auto consider = [&](int sk, int64_t tail_first) {
      consider_tile_plan(best, t, FP8_TILE_COSTS, M, N, (double)N * K, tiles, sk, tail_first, steps, cus, 1ll << 32);   // (32-bit offsets)
    };
    if (tn.fp8_split > 0) {
      consider(tn.fp8_split <= steps ? tn.fp8_split : steps, 0);
      continue;
    }
    // K in up to 8 parts of at least 8 steps, on up to 2.3 rounds of workgroups.  (All of 1 .. 8: without 5 and 7 4 % of the
    // problems had another plan, in the mean 1.3 % slower; 11776 x 576 at M = 1180 27.5 -> 22.5 us)
    for (int sk = 1; sk <= 8; ++sk)
      if (sk == 1 || (steps / sk >= 8 && tiles * sk * 10 <= cus * 23)) consider(sk, 0);
    // 256 x 256 tiles that end in a round of workgroups at most half full: the tiles of that round in parts of at least 16
    // steps that fill it, the others whole
    if (t.id == 1 && tiles > cus && rest > 0 && tn.exp[6] > 1) best = TilePlan();      // (development switch: this plan alone)
    if (t.id == 1 && tiles > cus && rest > 0 && tn.exp[10] != 1)
      for (int sk : {2, 3, 4})
        if (rest * sk <= cus && (tn.exp[6] > 1 ? sk == tn.exp[6] && steps / sk >= 4 : steps / sk >= 16)) consider(sk, tiles - rest);
  }
  if (best.id < 0) return best;      // an unknown shape was forced: the other kernels take the problem
  // A split K with compute units left for the parts of one more tile row: that row runs past M beside the real ones, as
  // with an unsplit K (see m_tiles_extra in dispatch_tile); its workgroups take no part in the hand-over, but tile
  // positions -- and with them the places in the scratch -- count it.  Cold: 7168 x 2048 at M = 40 / 64 / 192 12.1 / 13.6 /
  // 18.0 -> 10.3 / 10.4 / 12.8 us, 8192 x 1024 at M = 40 .. 192 12.4 .. 13.2 -> 10.7 .. 11.0 us.
  if (best.sk > 1 && best.tail_first == 0 && tn.exp[13] != 1) {
    const int64_t rows = (M + best.bm - 1) / best.bm, cols = best.tiles / rows;
    if (rows <= 3 && (best.tiles + cols) * best.sk <= cus) best.extra_tiles = cols;
  }
  return best;
}

static TilePlan plan_tile3(int M, int N, int K) {
  static thread_local TilePlanTable table;
  if (tuning_active()) return make_plan_tile3(M, N, K);
  return table.get(M, N, K, num_cus_current_device(), [&] { return make_plan_tile3(M, N, K); });
}

template <bool BF16_OUT>
static int dispatch_tile(const Fp8MMParams& p_in, int64_t c_tmp_bytes, int64_t counter_ints, hipStream_t s) {
  Fp8MMParams p = p_in;
  // Descriptors end with the last row and not a pitch behind its start: an operand may be the trailing columns of its storage, and the
  // 256 x 256 tile requests 128 bytes where K leaves 64.
  p.a_extent = (uint32_t)((int64_t)(p.M - 1) * p.lda + p.K);
  p.b_extent = (uint32_t)((int64_t)(p.N - 1) * p.ldb + p.K);
  // A step that ends past K: the offset of a chunk past K, 2 GiB, has to be past the operand's end, and its sum with a place in the operand may not wrap.
  const bool far = (uint64_t)(p.M - 1) * (uint64_t)p.lda + (uint64_t)p.K >= (1ull << 31) || (uint64_t)(p.N - 1) * (uint64_t)p.ldb + (uint64_t)p.K >= (1ull << 31);
  const bool direct_ok = tuning().fp8_tile_impl == 0 && (uint64_t)p.M * (uint64_t)p.lda < (1ull << 32) && (uint64_t)p.N * (uint64_t)p.ldb < (1ull << 32) &&
                         (p.K % 64 == 0 || !far);
  if (direct_ok && tuning().fp8_tile_impl == 0 && tuning().fp8_tile_cfg >= 0) {
    TilePlan pl = plan_tile3(p.M, p.N, p.K);
    const bool half_step = pl.id > 10 && p.K % 128 != 0;      // K ends inside a step of 128 bytes (the 256-wide tiles step by 64)
    if (half_step && far) pl.id -= 10;                        // (K % 64 = 0: the same tile by slices of 64 bytes)
    // without (enough) scratch from the caller the unsplit kernel still gives the result
    if (pl.sk > 1 && (p.c_tmp == nullptr || p.counters == nullptr || counter_ints < pl.counter_ints() ||
                      c_tmp_bytes < pl.tmp_bytes()))
      pl.sk = 1;
    if (pl.sk == 1) pl.tail_first = 0;
    p.SK = pl.sk;
    p.tail_first = (int)pl.tail_first;
    if (pl.id > 0) {
      const int64_t tiles_m = (p.M + pl.bm - 1) / pl.bm;
      const int64_t cus = num_cus_current_device();
      // (with K split over workgroups the rotation gains nothing on cold weights and costs 20-30 % on cached ones.)
      // Up to 4 tile rows on a device that the tiles leave a fifth empty; any number of tile rows in one round of workgroups
      // when the weights are small enough (32 MiB: 4 MiB per L2) that the part another tile row has just read is still in
      // the L2 -- cold, 4096 x 4096 at M = 256 .. 512: 16.2 / 23.5 -> 12.7 / 18.8 us, 4096 x 6144 at M = 1024 41.4 -> 36.4 us,
      // 2048 x 2048 at M = 1024 13.9 -> 11.2 us; larger weights lose (6656 x 6656 at M = 72: 17.3 -> 24.1 us; 4096 x 28672
      // at M = 192 .. 384: +7 %), and so do tiles that need a second round (4096 x 6144 at M = 768: 35.9 -> 41.6 us).
      p.rotate_k = pl.sk == 1 && tiles_m > 1 &&
                   ((tiles_m <= 4 && pl.tiles * 5 < cus * 4) || (pl.tiles <= cus && (int64_t)p.K * p.N <= ((int64_t)32 << 20)));
      // A last tile row filled to a third at most.  Two tile rows: nobody rotates (the nearly empty row finishes early
      // whatever it reads, and rotated it reads for nothing what the full row does not read with it; cold: 4096 x 4096 at
      // M = 66 .. 84 13.3 -> 11.1 .. 11.8 us, 4096 x 6144 13.7 -> 11.6 .. 12.5 us).  64 x 64 tiles: the same with three and
      // four rows (4096 x 4096 at M = 132 .. 144 13.2 -> 11.2 .. 11.9 us, at M = 196 .. 208 13.1 -> 11.5 .. 12.1 us; from a fill
      // of 24 rows on the rotation is level or ahead).  Larger tiles with three rows and more keep the rotation (64 x 128:
      // 4096 x 6144 at M = 132 19.5 against 21.2 us, 4096 x 4096 at M = 264 18.2 against 21.1 us).
      if (p.rotate_k == 1 && ((int64_t)p.M - (tiles_m - 1) * pl.bm) * 3 <= pl.bm && (tiles_m == 2 || pl.bn == 64)) p.rotate_k = 0;
      // one or two tile rows on a wide layer: by tile column instead (see the kernel)
      if (p.rotate_k == 0 && pl.sk == 1 && tiles_m <= 2 && pl.tiles * 5 >= cus * 2) p.rotate_k = 2;
      if (tuning().exp[12] == 1) p.rotate_k = 0;      // (development switch: every tile starts at the first K step)
      // A tile row past M.  With at most three tile rows and compute units to spare, one more row of workgroups runs
      // beside the real ones: its activation rows lie past M (see `load`; nothing is stored), its weight
      // loads are the real tiles' own.  Every weight line is then asked for by two workgroups on two compute units,
      // whichever gets there first, and arrives earlier for the other: what one compute unit has in flight is what bounds
      // a tile's operand stream at these sizes (deeper rings do not help, a second requester does).  Cold, 64 x 64 tiles:
      // 4096 x 4096 at M = 64 .. 192 13.2 .. 16.4 -> 10.8 .. 11.1 us, 5120 x 5120 at M = 64 / 128 17.0 / 17.4 -> 13.2 / 13.3 us,
      // 2048 x 2048 at M = 128 8.6 -> 7.3 us; 128 x 128 tiles: 4096 x 6144 at M = 384 25.8 -> 23.5 us, 8192 x 8192 at M = 384
      // 46.7 -> 41.7 us.  The real rows then start together (rotated they lose the gain); from four tile rows on the
      // rotation alone is level or ahead (3072 x 3072 at M = 384 14.8 against 16.0 us) and stays.
      p.m_tiles_extra = pl.extra_tiles > 0 && pl.sk > 1 ? 1 : 0;
      if (pl.sk == 1 && pl.tail_first == 0 && tiles_m <= 3 && pl.tiles + pl.tiles / tiles_m <= cus && tuning().exp[13] != 1) {
        p.m_tiles_extra = 1;
        p.rotate_k = 0;
      }
    }
    // All K that are no multiple of 64 once went through registers and padded LDS: 80 drawn problems of 33 .. 8192 rows take 0.56 of that time in the mean (126 rows of
    // 8400 x 4096 59.5 -> 22.0 us, 1700 of 5968 x 2368 52.4 -> 50.8); K % 128 = 64 went by slices of 64, half a cache line: 90 problems 0.95 (232 rows of 13632 x 25280
    // 163 -> 136 us, the worst 198 of 1472 x 5632 8.7 -> 9.2), and does so where an operand ends beyond 2 GiB.
    const bool tail = p.K % 64 != 0 || (half_step && !far);
    switch (tail ? -pl.id : pl.id) {
      case -1: return launch_tile3<BF16_OUT, 256, 256, 2, 4, 5, 1, 2, true>(p, s);
      case -13: return launch_tile3<BF16_OUT, 128, 128, 2, 4, 4, 2, 0, true>(p, s);
      case -14: return launch_tile3<BF16_OUT, 64, 128, 2, 2, 5, 2, 0, true>(p, s);
      case -15: return launch_tile3<BF16_OUT, 64, 64, 2, 2, 5, 2, 0, true>(p, s);
      case -16: return launch_tile3<BF16_OUT, 128, 64, 2, 2, 5, 2, 0, true>(p, s);
      case -17: return launch_tile3<BF16_OUT, 128, 256, 2, 4, 3, 2, 0, true>(p, s);
      case -19: return launch_tile3<BF16_OUT, 256, 128, 4, 2, 3, 2, 0, true>(p, s);
      case 1: return launch_tile3<BF16_OUT, 256, 256, 2, 4, 5, 1, 2>(p, s);    // alternating phases, slices requested in pairs (see the kernel)
      case 10: return launch_tile3<BF16_OUT, 256, 384, 2, 4, 4, 1, 1>(p, s);   // 8 wavefronts of 128 x 96, alternating phases, one slice at a time
      // two k-slices per step
      case 13: return launch_tile3<BF16_OUT, 128, 128, 2, 4, 4, 2>(p, s);
      case 14: return launch_tile3<BF16_OUT, 64, 128, 2, 2, 5, 2>(p, s);
      case 15: return launch_tile3<BF16_OUT, 64, 64, 2, 2, 5, 2>(p, s);
      case 16: return launch_tile3<BF16_OUT, 128, 64, 2, 2, 5, 2>(p, s);
      case 17: return launch_tile3<BF16_OUT, 128, 256, 2, 4, 3, 2>(p, s);
      case 19: return launch_tile3<BF16_OUT, 256, 128, 4, 2, 3, 2>(p, s);
      // one
      case 3: return launch_tile3<BF16_OUT, 128, 128, 2, 4, 5>(p, s);
      case 4: return launch_tile3<BF16_OUT, 64, 128, 2, 2, 5>(p, s);
      case 5: return launch_tile3<BF16_OUT, 64, 64, 2, 2, 5>(p, s);
      case 6: return launch_tile3<BF16_OUT, 128, 64, 2, 2, 5>(p, s);
      case 7: return launch_tile3<BF16_OUT, 128, 256, 2, 4, 5>(p, s);
      case 9: return launch_tile3<BF16_OUT, 256, 128, 4, 2, 5>(p, s);
      default: break;
    }
  }
  p.SK = 1;
  if (direct_ok && p.K % F8_BK == 0) {
    const int cus2 = num_cus_current_device();
    auto tiles2 = [&](int bm, int bn) { return (int64_t)((p.M + bm - 1) / bm) * ((p.N + bn - 1) / bn); };
    if (tiles2(256, 256) >= cus2) return launch_tile2<BF16_OUT, 4, 4>(p, s);
    if (tiles2(128, 128) >= cus2) return launch_tile2<BF16_OUT, 2, 2>(p, s);
    return launch_tile2<BF16_OUT, 1, 2>(p, s);
  }
  const int cus = num_cus_current_device();
  auto tiles = [&](int bm, int bn) { return (int64_t)((p.M + bm - 1) / bm) * ((p.N + bn - 1) / bn); };
  if (tiles(256, 256) >= cus) return launch_tile<BF16_OUT, 4, 4>(p, s);
  if (tiles(128, 128) >= cus) return launch_tile<BF16_OUT, 2, 2>(p, s);
  return launch_tile<BF16_OUT, 1, 2>(p, s);
}

template <bool BF16_OUT, int KS, int MB, bool HALVES = false>
static void launch_stream(const Fp8MMParams& p_in, int wk, int gx, hipStream_t s) {
  Fp8MMParams p = p_in;
  p.nt_base = (p.N / 16) / gx;
  p.nt_rem = (p.N / 16) % gx;
  p.a_extent = (uint32_t)((int64_t)(p.M - 1) * p.lda + p.K);
  p.b_extent = (uint32_t)((int64_t)(p.N - 1) * p.ldb + p.K);
  const size_t lds = wk > 1 ? (size_t)2 * wk * MB * 64 * sizeof(v4f) : 0;
  if (p.nt_base == 1 && p.nt_rem == 0)
    launch_fp8_stream(fp8_mm_stream_kernel<BF16_OUT, KS, MB, HALVES, false>, dim3(gx, HALVES ? 2 : 1), wk, lds, s, p);
  else
    launch_fp8_stream(fp8_mm_stream_kernel<BF16_OUT, KS, MB, HALVES, true>, dim3(gx, HALVES ? 2 : 1), wk, lds, s, p);
}

// The stream kernel addresses its operands with 32-bit offsets from buffer descriptors: both must end below 2 GiB
// (otherwise the tile kernels take the problem).
static bool stream_offsets_fit(const Fp8MMParams& p) {
  return (int64_t)(p.M - 1) * p.lda + p.K < (1ll << 31) && (int64_t)(p.N - 1) * p.ldb + p.K < (1ll << 31);
}

// K steps (of 128) per wavefront of the stream kernel for a problem, 0 if the kernel does not take it (the activations of
// a wavefront's K slab live in registers: at most 8 wavefronts along K, 14 steps each for one m-block, 8 for two).
static int stream_steps_per_wave(int64_t M, int64_t N, int64_t K) {
  const int64_t steps = (K + 127) / 128;
  // three and four m-blocks: K = 1664 .. 4096 (4 steps per wavefront keep the registers, and the workgroup must have a
  // wavefront per m-block for the reduction).  The time of the tile kernel over this one's, geometric means over 3093 random
  // problems, cold:                 K 1665-2560   2561-3072   3073-3584   3585-4096
  //   M 33 .. 48, N <= 4096          1.29 - 1.51   1.16 - 1.42  1.03 - 1.27  0.95 - 1.12
  //   M 33 .. 48, N 4097 .. 8192     1.02 - 1.16   1.03 - 1.13  1.04 - 1.11  0.91 - 1.04
  //   M 49 .. 64, N <= 4096          1.08 - 1.34   0.96 - 1.28  0.87 - 1.19  0.82 - 0.93
  // and 0.79 .. 1.05 on wider layers.  (2048 x 960 at M = 49 7.1 -> 6.0 us, 1664 x 4992 at M = 34 6.9 -> 6.4 us)
  if (M > 32) {
    if (M > 64 || steps < 13 || steps > 8 * 4) return 0;
    if (tuning().fp8_path == 1) return 4;
    return M <= 48 ? (N <= (steps <= 28 ? 8192 : 4096) ? 4 : 0) : (N <= 4096 && steps <= (M <= 56 ? 24 : 20) ? 4 : 0);
  }
  if (steps <= 8 * 4) return 4;
  if (steps <= 8 * 8) return 8;
  if (steps <= 8 * 14 && M <= 16) return 14;
  return 0;
}

// The stream kernel over two halves of K (two workgroups per n-tile range, partial tiles handed over through the caller's
// scratch): K steps per wavefront, 0 if this route does not take the problem.  It covers what the registers of one
// workgroup cannot at two m-blocks: 16 < M <= 32 up to K = 16384, on layers whose workgroups fit the device at once (cold
// against the tile kernel with K split: 9728 x 1152 at M = 17 11.0 against 11.9 us, 10112 x 1920 at M = 27 12.4 against 13.5 us; on
// wider ones the tiles are ahead, 12544 x 2560 at M = 17 15.2 against 19.6 us, 8320 x 9920 at M = 22 23.0 against 32.2 us).
static int stream_split_steps_per_wave(int64_t M, int64_t N, int64_t K) {
  if (tuning().fp8_stream_split < 0 || M <= 16 || M > 32 || stream_steps_per_wave(M, N, K) != 0 ||
      N / 8 > num_cus_current_device())
    return 0;
  const int64_t half = ((K + 127) / 128 + 1) / 2;
  return half <= 8 * 8 ? 8 : 0;
}

template <bool BF16_OUT>
static bool dispatch_stream_split(const Fp8MMParams& p, int64_t c_tmp_bytes, int64_t counter_ints, hipStream_t s) {
  const int ks = stream_split_steps_per_wave(p.M, p.N, p.K);
  if (ks == 0 || !stream_offsets_fit(p)) return false;
  const int MB = (p.M + 15) / 16, NT = p.N / 16;
  if (p.c_tmp == nullptr || p.counters == nullptr || counter_ints < (int64_t)NT * MB ||
      c_tmp_bytes < (int64_t)2 * NT * MB * 1024 || (int64_t)2 * NT * MB * 1024 >= (1ll << 31))
    return false;                                   // without the scratch the tile kernel still gives the result
  const int half = ((p.K + 127) / 128 + 1) / 2;
  const int wk = (half + ks - 1) / ks;              // >= 5: the K range of this route starts above one workgroup's
  const int cus = num_cus_current_device();
  const int rounds = (2 * NT + cus - 1) / cus;
  int gx = tuning().fp8_gx > 0 ? tuning().fp8_gx : (NT + rounds - 1) / rounds;
  if (gx > NT) gx = NT;
  launch_stream<BF16_OUT, 8, 2, true>(p, wk, gx, s);
  return true;
}

template <bool BF16_OUT, int KS, int MB, int NSR>
static bool launch_stream2(const Fp8MMParams& p_in, int wk, int gx, hipStream_t s) {
  Fp8MMParams p = p_in;
  p.nt_base = (p.N / 16) / gx;
  p.nt_rem = (p.N / 16) % gx;
  p.a_extent = (uint32_t)((int64_t)(p.M - 1) * p.lda + p.K);
  p.b_extent = (uint32_t)((int64_t)(p.N - 1) * p.ldb + p.K);
  const size_t lds = (size_t)wk * NSR * 4096 + (wk > 1 ? (size_t)2 * wk * MB * 64 * sizeof(v4f) : 0);
  auto kern = fp8_mm_stream2_kernel<BF16_OUT, KS, MB, NSR>;
  static size_t reserved[VAQ_MAX_DEVICES];
  if (reserve_dynamic_lds(reinterpret_cast<const void*>(kern), lds, reserved, "fp8_scaled_mm") != VAQ_OK) return false;      // (the kernel above then takes the problem)
  launch_fp8_stream(kern, dim3(gx), wk, lds, s, p);
  return true;
}

// Steps per wavefront of the stream kernel with the weights through LDS, 0 where the kernel above stays.  From 13500 problems
// drawn over M = 1 .. 32, K = 1024 .. 16384, N = 1024 .. 28672 with cold weights, every choice timed:
//  * up to 16 rows: 4 steps up to K = 1536 (2-7 % ahead of 8), 8 up to K = 3584, 16 beyond.  Fewer wavefronts with longer
//    streams: against 8 steps -10 .. -14 % at K = 2500 .. 3072, -1 .. -6 % to 3584, level to 3840, +1.5 % to 4096 (9356 problems),
//    6-8 % at K = 4100 .. 8192 (M = 1 / 4 / 16, us, against the kernel above:
//    4096 x 6144 8.6 / 9.0 / 10.3 -> 6.6 / 6.7 / 7.2, 4096 x 28672 25.8 / 26.1 / 27.8 -> 19.4 / 19.6 / 20.6, 14336 x 4096 13.8 /
//    14.8 / 18.0 -> 12.0 / 12.4 / 15.3);
//  * two m-blocks: 4 steps up to K = 1536 (4 % ahead), 8 to K = 8192 (3-7 % ahead of 4; against the kernel above, M = 24 / 32:
//    5120 x 5120 13.9 / 14.7 -> 10.9 / 11.8 us, 8192 x 8192 20.9 / 22.3 -> 19.4 / 20.7 us); 16 do not fit the registers.
// (development switch exp[4]: 1 / 2 / 3 force 8 / 4 / 16 steps, 9 switches the kernel off)
static int stream2_steps_per_wave(const Fp8MMParams& p) {
  const int sw = tuning().exp[4];
  if (sw == 9 || p.M > 32 || p.K % 16 != 0 || !stream_offsets_fit(p)) return 0;
  const int steps = (p.K + 127) / 128, MB = (p.M + 15) / 16;
  int ks = 0;
  if (sw >= 1 && sw <= 3) ks = sw == 1 ? 8 : (sw == 2 ? 4 : 16);
  else if (MB == 1) ks = steps <= 12 ? 4 : (steps <= 28 ? 8 : (steps <= 128 ? 16 : 0));
  else ks = steps <= 12 ? 4 : (steps <= 64 ? 8 : 0);
  if (ks == 0 || (steps + ks - 1) / ks > 8 || (MB == 2 && ks == 16)) return 0;
  return ks;
}

template <bool BF16_OUT>
static bool dispatch_stream2(const Fp8MMParams& p, hipStream_t s) {
  const int ks = stream2_steps_per_wave(p);
  if (ks == 0) return false;
  const int steps = (p.K + 127) / 128;
  const int wk = (steps + ks - 1) / ks;
  const int MB = (p.M + 15) / 16, NT = p.N / 16;
  const int cus = num_cus_current_device();
  const int rounds = (NT + cus - 1) / cus;
  int gx = (NT + rounds - 1) / rounds;
  // one workgroup per compute unit, except that a short K (a workgroup of one to three wavefronts) takes two on a layer of
  // more than three rounds (K <= 1536: 8 % ahead at 769 .. 1024 n-tiles, longer K 3-15 % behind)
  if (MB == 1 && steps <= 12 && NT > 3 * cus) gx = 2 * cus;
  if (tuning().fp8_gx > 0) gx = tuning().fp8_gx;
  if (gx > NT) gx = NT;
  if (MB == 1) {
    if (ks == 4) return launch_stream2<BF16_OUT, 4, 1, 2>(p, wk, gx, s);
    if (ks == 8) return launch_stream2<BF16_OUT, 8, 1, 4>(p, wk, gx, s);
    return launch_stream2<BF16_OUT, 16, 1, 4>(p, wk, gx, s);
  }
  if (ks == 4) return launch_stream2<BF16_OUT, 4, 2, 2>(p, wk, gx, s);
  return launch_stream2<BF16_OUT, 8, 2, 4>(p, wk, gx, s);
}

template <bool BF16_OUT>
static bool dispatch_stream(const Fp8MMParams& p, hipStream_t s) {
  const int steps = (p.K + 127) / 128;
  const int MB = (p.M + 15) / 16;
  const int ks = stream_steps_per_wave(p.M, p.N, p.K);
  if (ks == 0 || !stream_offsets_fit(p)) return false;
  const int wk = (steps + ks - 1) / ks;
  const int NT = p.N / 16;
  // one workgroup per compute unit, the n-tiles dealt out evenly over the fewest rounds: every workgroup loads all the
  // activations of its K slabs, so more workgroups than compute units only multiply that traffic (measured, cold weights,
  // against two workgroups per compute unit: 4096 x 6144 at M = 16 / 32 11.9 / 16.4 -> 10.4 / 12.4 us, 4096 x 28672
  // 31.8 / 38.0 -> 30.4 / 31.9 us, M = 1 unchanged or 3 % faster)
  const int cus = num_cus_current_device();
  const int rounds = (NT + cus - 1) / cus;
  int gx = (NT + rounds - 1) / rounds;
  // One m-block, measured with cold weights: on a layer of many rounds two workgroups per compute unit are ahead
  // (4096 x 28672 at M = 1 / 4 / 16: 28.1 / 28.2 / 29.2 -> 25.7 / 26.1 / 27.8 us; at M = 32 30.5 -> 33.0 us), and with up to
  // four rows a layer of one to two rounds runs one tile per workgroup (4096 x 6144 at M = 1 / 4: 9.3 / 9.4 -> 8.6 / 9.0 us;
  // at M = 16 10.2 -> 10.9 us).
  if (MB == 1 && NT >= 4 * cus) gx = 2 * cus;
  else if (p.M <= 4 && NT > cus && NT <= 2 * cus) gx = NT;
  if (tuning().fp8_gx > 0) gx = tuning().fp8_gx;
  if (gx > NT) gx = NT;
  if (MB == 1) {
    if (ks == 4) launch_stream<BF16_OUT, 4, 1>(p, wk, gx, s);
    else if (ks == 8) launch_stream<BF16_OUT, 8, 1>(p, wk, gx, s);
    else launch_stream<BF16_OUT, 14, 1>(p, wk, gx, s);
  } else if (MB == 2) {
    if (ks == 4) launch_stream<BF16_OUT, 4, 2>(p, wk, gx, s);
    else launch_stream<BF16_OUT, 8, 2>(p, wk, gx, s);
  } else if (MB == 3) {
    launch_stream<BF16_OUT, 4, 3>(p, wk, gx, s);
  } else {
    launch_stream<BF16_OUT, 4, 4>(p, wk, gx, s);
  }
  return true;
}

// Whether the kernel of fp8_regs_kernel.h takes a problem: where its price is 7 % below that of the tile plan, or not so far above that of the stream kernel with
// weights through LDS -- its rows' activations, its n-tiles in rounds of one to a compute unit, the weights from memory; fitted to 291 of the timings
// below, 7 % rms.  Up to 16 rows 3 %; from 17 rows on, which the price counts as 32 whatever their number, 10 % up to N = 12288 and none beyond, where the stream kernel
// is at memory speed (2944 x 21248 at M = 20 12.4 us, 15.2 here).  At 3 % below throughout 8192 x 8192 at M = 24 stayed there for 22.7 us, 12.9 here.  (33 .. 64 rows
// where the other stream kernel was ahead of the tiles: 20 of 20 problems faster here, 0.70 of the time.)  Not up to 4 rows, where it is ahead by 2 % of the time
// where at all.  811 timed problems: takes 0.71 / 0.88 / 0.68 / 0.52 / 0.32 of those of 5 .. 16 / .. 32 / .. 64 / .. 128 / .. 256
// rows, for 0.95 / 0.84 / 0.77 / 0.80 / 0.86 of the time, 2 % of them more than 3 % slower.  901 calls of other drawn layers 0.915 of their time at the first shares, 600
// of 5 .. 32 rows another 0.990 from those to these (14208 x 4608 at M = 32 17.4 -> 19.7 us, 2304 x 12800 at M = 16 7.2 -> 7.7).
static bool takes_regs(int M, int N, int K, Fp8RegsPlan* plan, double* other) {
  *plan = fp8_regs_plan(M, N, K);
  const int steps = (K + 127) / 128;
  if (M <= 32 && steps <= (M <= 16 ? 128 : 64)) {      // (stream2_steps_per_wave)
    const double k = K / 1024.0, act = 0.349 * M / 16 * k * (1 + 0.0311 * k), rounds = ceil(N / 16.0 / num_cus_current_device());
    const double core = 0.372 * rounds * k + act, mem = 0.137e-6 * K * N;
    *other = 2.3 + cbrt(core * core * core + mem * mem * mem) + 0.304 * 2e-6 * M * N;
    // (17 .. 32 rows of K 1537 .. 3072: 0.98.  378 problems of K 1024 .. 6144, both timed: at 1.1 throughout the choice takes 1.0078 of the faster one's time and 44 calls here are more than 3 %
    // slower, 27 of them on that K (2976 x 10240 at M = 22 9.6 us, 8.4 there; 2064 x 7104 at M = 30 6.4, 5.8); so 1.0049 and 25.)
    return M > 4 && plan->us < (M <= 16 ? 1.03 : N > 12288 ? 1.0 : K > 1536 && K <= 3072 ? 0.98 : 1.1) * *other;
  }
  *other = plan_tile3(M, N, K).us;
  return M > 4 && plan->us < 0.93 * *other;
}

// The same for a call, from a table per thread.  A switch that names another kernel or a plan of one keeps it out; exp[11]: 1 never, else its plan, n-tiles |
// m-blocks << 4.
static bool fp8_regs_chosen(int M, int N, int K, int* mb, int* j) {
  const VaqTuning& tn = tuning();
  if (tn.exp[11] > 1) {
    *mb = tn.exp[11] >> 4;
    *j = tn.exp[11] & 15;
    return true;
  }
  if (tn.exp[11] == 1 || tn.fp8_path > 0 || tn.fp8_tile_impl != 0 || tn.fp8_tile_cfg != 0 || tn.fp8_split > 0 || tn.fp8_gx > 0 || tn.exp[4] > 0 || tn.exp[6] > 0 ||
      tn.exp[12] > 0 || tn.exp[13] > 0)
    return false;
  static thread_local PlanTable<int> table;
  const int at = table.get(M, N, K, num_cus_current_device(), [&] {
    const TuningScope automatic(nullptr);
    Fp8RegsPlan plan;
    double other = 0;
    return takes_regs(M, N, K, &plan, &other) ? plan.j | plan.mb << 4 : 0;
  });
  *mb = at >> 4;
  *j = at & 15;
  return at != 0;
}

}  // namespace vaq

extern "C" int vaq_fp8_regs_plan(int64_t size_m, int64_t size_n, int64_t size_k, double* plan) {
  using namespace vaq;
  VAQ_CHECK_ARG(size_m > 0 && size_m <= FP8_REGS_MAX_M && size_n > 0 && size_n % 16 == 0 && size_k > 0 && size_k % 16 == 0 && size_n < (1 << 24) &&
                    size_k < (1 << 24) && plan != nullptr, "fp8_regs_plan: bad arguments");
  Fp8RegsPlan r;
  plan[4] = takes_regs((int)size_m, (int)size_n, (int)size_k, &r, &plan[3]) ? 1 : 0;
  plan[0] = r.j;
  plan[1] = r.mb;
  plan[2] = r.us;
  return VAQ_OK;
}

extern "C" int vaq_fp8_scaled_mm_workspace(int64_t size_m, int64_t size_n, int64_t size_k, size_t* c_tmp_bytes,
                                           size_t* counter_ints) {
  return vaq_fp8_scaled_mm_workspace_tuned(size_m, size_n, size_k, c_tmp_bytes, counter_ints, nullptr);
}

extern "C" int vaq_fp8_scaled_mm_workspace_tuned(int64_t size_m, int64_t size_n, int64_t size_k, size_t* c_tmp_bytes,
                                                 size_t* counter_ints, const VaqTuning* tuning_or_null) {
  using namespace vaq;
  const TuningScope scope(tuning_or_null);
  VAQ_CHECK_ARG(c_tmp_bytes && counter_ints, "fp8_scaled_mm_workspace: null output pointer");
  VAQ_CHECK_ARG(size_m >= 0 && size_n > 0 && size_k > 0 && size_m < (1ll << 31) && size_n < (1ll << 31) &&
                    size_k < (1ll << 31), "fp8_scaled_mm_workspace: bad shape M=%lld N=%lld K=%lld", (long long)size_m,
                (long long)size_n, (long long)size_k);
  *c_tmp_bytes = 0;
  *counter_ints = 0;
  const bool stream = tuning().fp8_path != 2 && stream_steps_per_wave(size_m, size_n, size_k) != 0;      // needs no scratch
  if (stream) return VAQ_OK;
  if (tuning().fp8_path != 2 && stream_split_steps_per_wave(size_m, size_n, size_k) != 0) {
    const size_t units = (size_t)(size_n / 16) * (size_t)((size_m + 15) / 16);
    *c_tmp_bytes = 2 * units * 1024;
    *counter_ints = units;
    return VAQ_OK;
  }
  if (tuning().fp8_tile_impl != 0 || tuning().fp8_tile_cfg < 0) return VAQ_OK;
  const TilePlan pl = plan_tile3((int)size_m, (int)size_n, (int)size_k);
  *c_tmp_bytes = (size_t)pl.tmp_bytes();
  *counter_ints = (size_t)pl.counter_ints();
  return VAQ_OK;
}

extern "C" int vaq_fp8_scaled_mm(const uint8_t* a, int64_t lda, const uint8_t* b, int64_t ldb, const float* sa,
                                 int64_t sa_count, const float* sb, int64_t sb_count, const void* bias, void* out,
                                 int64_t ldc, int out_dtype, int64_t size_m, int64_t size_n, int64_t size_k,
                                 void* stream) {
  return vaq_fp8_scaled_mm_ws(a, lda, b, ldb, sa, sa_count, sb, sb_count, bias, out, ldc, out_dtype, size_m, size_n,
                              size_k, nullptr, 0, nullptr, 0, stream);
}

extern "C" int vaq_fp8_scaled_mm_ws(const uint8_t* a, int64_t lda, const uint8_t* b, int64_t ldb, const float* sa,
                                    int64_t sa_count, const float* sb, int64_t sb_count, const void* bias, void* out,
                                    int64_t ldc, int out_dtype, int64_t size_m, int64_t size_n, int64_t size_k,
                                    float* c_tmp, int64_t c_tmp_bytes, int32_t* counters, int64_t counter_ints,
                                    void* stream) {
  return vaq_fp8_scaled_mm_ws_tuned(a, lda, b, ldb, sa, sa_count, sb, sb_count, bias, out, ldc, out_dtype, size_m, size_n,
                                    size_k, c_tmp, c_tmp_bytes, counters, counter_ints, stream, nullptr);
}

extern "C" int vaq_fp8_scaled_mm_ws_tuned(const uint8_t* a, int64_t lda, const uint8_t* b, int64_t ldb, const float* sa,
                                          int64_t sa_count, const float* sb, int64_t sb_count, const void* bias,
                                          void* out, int64_t ldc, int out_dtype, int64_t size_m, int64_t size_n,
                                          int64_t size_k, float* c_tmp, int64_t c_tmp_bytes, int32_t* counters,
                                          int64_t counter_ints, void* stream, const VaqTuning* tuning_or_null) {
  using namespace vaq;
  const TuningScope scope(tuning_or_null);
  VAQ_CHECK_ARG(size_m >= 0 && size_n > 0 && size_k > 0, "fp8_scaled_mm: bad shape M=%lld N=%lld K=%lld",
                (long long)size_m, (long long)size_n, (long long)size_k);
  VAQ_CHECK_ARG(size_m < (1ll << 31) && size_n < (1ll << 31) && size_k < (1ll << 31), "fp8_scaled_mm: shape too large");
  VAQ_CHECK_ARG(size_k % 16 == 0 && size_n % 16 == 0, "fp8_scaled_mm: K = %lld and N = %lld must be multiples of 16",
                (long long)size_k, (long long)size_n);
  VAQ_CHECK_ARG(lda >= size_k && lda % 16 == 0, "fp8_scaled_mm: a row stride %lld must be >= K and a multiple of 16",
                (long long)lda);
  VAQ_CHECK_ARG(ldb >= size_k && ldb % 16 == 0, "fp8_scaled_mm: b column stride %lld must be >= K and a multiple of 16",
                (long long)ldb);
  VAQ_CHECK_ARG(ldc >= size_n && ldc % 8 == 0, "fp8_scaled_mm: out row stride %lld must be >= N and a multiple of 8",
                (long long)ldc);
  VAQ_CHECK_ARG(sa_count == 1 || sa_count == size_m, "fp8_scaled_mm: a_scales count %lld must be 1 or M",
                (long long)sa_count);
  VAQ_CHECK_ARG(sb_count == 1 || sb_count == size_n, "fp8_scaled_mm: b_scales count %lld must be 1 or N",
                (long long)sb_count);
  VAQ_CHECK_ARG(out_dtype == VAQ_F16 || out_dtype == VAQ_BF16, "fp8_scaled_mm: out dtype tag %d", out_dtype);
  if (size_m == 0) return VAQ_OK;
  VAQ_CHECK_ARG(a && b && sa && sb && out, "fp8_scaled_mm: null pointer");
  VAQ_CHECK_ARG(((uintptr_t)a % 16) == 0 && ((uintptr_t)b % 16) == 0 && ((uintptr_t)out % 8) == 0,
                "fp8_scaled_mm: a and b must be 16-byte aligned, out 8-byte aligned");
  VAQ_CHECK_ARG(((uintptr_t)sb % 16) == 0 && (!bias || ((uintptr_t)bias % 8) == 0),
                "fp8_scaled_mm: b_scales must be 16-byte aligned, bias 8-byte aligned");
  Fp8MMParams p;
  p.a = a; p.lda = lda; p.b = b; p.ldb = ldb;
  p.sa = sa; p.sa_per_row = (sa_count > 1 || size_m == 1) ? 1 : 0;
  p.sb = sb; p.sb_per_col = (sb_count > 1 || size_n == 1) ? 1 : 0;
  p.bias = (const uint16_t*)bias;
  p.out = (uint16_t*)out; p.ldc = ldc;
  p.M = (int)size_m; p.N = (int)size_n; p.K = (int)size_k;
  p.c_tmp = c_tmp;
  p.counters = counters;
  VAQ_CHECK_ARG(c_tmp == nullptr || ((uintptr_t)c_tmp % 16) == 0, "fp8_scaled_mm: c_tmp must be 16-byte aligned");
  hipStream_t s = (hipStream_t)stream;
  const bool bf16 = out_dtype == VAQ_BF16;
  bool done = false;
  const bool want_stream = tuning().fp8_path != 2 && stream_steps_per_wave(size_m, size_n, size_k) != 0;
  if (size_m <= FP8_REGS_MAX_M && size_n < (1 << 24) && size_k < (1 << 24) && stream_offsets_fit(p)) {
    int mb = 0, j = 0;
    if (fp8_regs_chosen(p.M, p.N, p.K, &mb, &j)) done = fp8_regs_launch(p, bf16, mb, j, s);
  }
  if (!done && tuning().fp8_path != 2) done = bf16 ? dispatch_stream2<true>(p, s) : dispatch_stream2<false>(p, s);
  if (!done && want_stream) done = bf16 ? dispatch_stream<true>(p, s) : dispatch_stream<false>(p, s);
  if (!done && tuning().fp8_path != 2)
    done = bf16 ? dispatch_stream_split<true>(p, c_tmp_bytes, counter_ints, s)
                : dispatch_stream_split<false>(p, c_tmp_bytes, counter_ints, s);
  if (!done) {
    int rc = bf16 ? dispatch_tile<true>(p, c_tmp_bytes, counter_ints, s) : dispatch_tile<false>(p, c_tmp_bytes, counter_ints, s);
    if (rc != VAQ_OK) return rc;
  }
  VAQ_CHECK_LAUNCH("fp8_scaled_mm");
  return VAQ_OK;
}
