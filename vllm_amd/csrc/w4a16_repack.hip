// GPTQ / AWQ int4 weight repack for gfx950.
//
// Input : GPTQ checkpoint tensor int32 [K/8, N]; word (r, n) holds codes of rows 8r..8r+7 of column n, row 8r+e in
//         bits [4e, 4e+4);
//         or AWQ (AutoAWQ) checkpoint tensor int32 [K, N/8]; word (k, c) holds the codes of row k, columns 8c..8c+7,
//         column 8c + {0,2,4,6,1,3,5,7}[p] in nibble position p.
// Output: int32 [K/16, 2N] (same byte count) in one of two orders.
//
//  NATIVE (what the GEMM kernels stream)
//    The matrix is cut into tiles of 128 rows (k) x 16 columns (n); tile (kt, nt) is the 1 KiB block number
//    nt * (K/128) + kt: the tiles of one 16-column strip are contiguous along K, so a wavefront that walks K for its
//    strip reads one sequential stream (measured: strided 1 KiB reads cost ~1.6x against sequential ones).
//    Inside a tile, lane L = 16*o + r (o = 0..3, r = 0..15) of a 64-wide wavefront owns the
//    16 bytes at offset 16*L: four words j = 0..3, word j holding the 8 codes of rows
//        k = 128*kt + 32*j + 8*o + e  (e = 0..7),  column n = 16*nt + r,
//    with code e stored in nibble position p where {0,2,4,6,1,3,5,7}[p] == e.  One 16-byte load per lane therefore
//    yields the A operands (row = n, 8 consecutive k per lane) of four v_mfma_f32_16x16x32 instructions that together
//    cover one quantisation group of 128 rows, and `(w >> 4i) & 0x000f000f | EX` produces operand register i directly.
//
//  MARLIN (bit-exact with the reference's gptq_marlin_repack, kept for the parity contract)
//    16 x 64 tiles; output word (kt*(N/64) + nt)*128 + th*4 + warp, th = 0..31, warp = 0..3, holds codes of rows
//    16*kt + 2*(th%4) + {0,1,8,9} for column 64*nt + 16*warp + th/4 (first four) and that column + 8 (last four),
//    nibble order {0,2,4,6,1,3,5,7}.
//
// 8-bit codes (GPTQ int32 [K/4, N], row 4r+e in bits [8e, 8e+8)) go to int32 [K/16, 4N]:
//  NATIVE  two 4-bit planes per tile: block 2*(nt*(K/128)+kt) holds the high nibbles (code >> 4) of the tile in the
//          order above, the next block the low nibbles, so the 4-bit kernels' dequantisation applies to each plane.
//  MARLIN  16 x 64 tiles of 256 words; words th*8 + warp*2 + {0, 1} hold, one byte each, rows 16*kt + 2*(th%4) +
//          {0, 8, 1, 9} of column 64*nt + 16*warp + th/4 (word 0) and that column + 8 (word 1).
//  NATIVE_BYTES (FP8 e4m3 weights, whose codes are not linear in their bits, so the nibble planes are of no use): per
//          tile two 1 KiB blocks; block h (0 / 1) gives lane L = 16*o + r the 16 bytes of rows 128*kt + 32*j + 8*o + e,
//          j = 2h (bytes 0..7, e = byte index) and j = 2h + 1 (bytes 8..15), column 16*nt + r: every 8 bytes are the A
//          operand of one v_mfma_f32_16x16x32 after four packed FP8 -> 16-bit conversions.
//
// With `perm` (act_order sort indices) output row k takes input row perm[k].
#include "vaq_common.h"

namespace vaq {

__device__ inline uint32_t fetch_code(const uint32_t* __restrict__ qw, const int32_t* __restrict__ perm, int64_t k,
                                      int64_t n, int64_t size_n) {
  int64_t src = perm ? (int64_t)perm[k] : k;
  uint32_t word = qw[(src >> 3) * size_n + n];
  return (word >> ((src & 7) * 4)) & 0xFu;
}

// AWQ source: nibble position of column n inside its word is {0,4,1,5,2,6,3,7}[n % 8] (the inverse of the AutoAWQ
// interleave {0,2,4,6,1,3,5,7}); reference: awq_marlin_repack.cu:95-103.
__device__ inline uint32_t fetch_code_awq(const uint32_t* __restrict__ qw, int64_t k, int64_t n, int64_t size_n) {
  const uint32_t word = qw[k * (size_n >> 3) + (n >> 3)];
  const int pos = (int)(((n & 1) << 2) | ((n & 7) >> 1));
  return (word >> (pos * 4)) & 0xFu;
}

__device__ inline uint32_t fetch_code8(const uint32_t* __restrict__ qw, const int32_t* __restrict__ perm, int64_t k,
                                       int64_t n, int64_t size_n) {
  int64_t src = perm ? (int64_t)perm[k] : k;
  uint32_t word = qw[(src >> 2) * size_n + n];
  return (word >> ((src & 3) * 8)) & 0xFFu;
}

__device__ inline uint32_t interleave_pack(const uint32_t v[8]) {
  // nibble position p <- element {0,2,4,6,1,3,5,7}[p]
  return v[0] | (v[2] << 4) | (v[4] << 8) | (v[6] << 12) | (v[1] << 16) | (v[3] << 20) | (v[5] << 24) | (v[7] << 28);
}

// One thread per output word; native layout.
template <bool HAS_PERM, bool AWQ>
__global__ __launch_bounds__(256) void repack_native_kernel(const uint32_t* __restrict__ qw,
                                                             const int32_t* __restrict__ perm,
                                                             uint32_t* __restrict__ out, int64_t size_k,
                                                             int64_t size_n) {
  const int64_t total = size_k * size_n / 8;
  const int64_t k_tiles = size_k / 128;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int j = idx & 3;
    const int lane = (idx >> 2) & 63;
    const int64_t tile = idx >> 8;
    const int64_t nt = tile / k_tiles, kt = tile - nt * k_tiles;
    const int o = lane >> 4, r = lane & 15;
    const int64_t k0 = kt * 128 + j * 32 + o * 8;
    const int64_t n = nt * 16 + r;
    uint32_t res;
    if constexpr (AWQ) {
      uint32_t v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = fetch_code_awq(qw, k0 + e, n, size_n);
      res = interleave_pack(v);
    } else if constexpr (HAS_PERM) {
      uint32_t v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = fetch_code(qw, perm, k0 + e, n, size_n);
      res = interleave_pack(v);
    } else {
      // the 8 codes are exactly one input word; only the nibble order changes
      const uint32_t w = qw[(k0 >> 3) * size_n + n];
      uint32_t v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (w >> (4 * e)) & 0xFu;
      res = interleave_pack(v);
    }
    out[idx] = res;
  }
}

// One thread per output word; reference (Marlin) order.
template <bool AWQ>
__global__ __launch_bounds__(256) void repack_marlin_kernel(const uint32_t* __restrict__ qw,
                                                             const int32_t* __restrict__ perm,
                                                             uint32_t* __restrict__ out, int64_t size_k,
                                                             int64_t size_n) {
  const int64_t total = size_k * size_n / 8;
  const int64_t n_tiles = size_n / 64;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int warp = idx & 3;
    const int th = (idx >> 2) & 31;
    const int64_t tile = idx >> 7;
    const int64_t kt = tile / n_tiles, nt = tile - kt * n_tiles;
    const int64_t n = nt * 64 + warp * 16 + (th >> 2);
    const int64_t kbase = kt * 16 + (th & 3) * 2;
    const int off[4] = {0, 1, 8, 9};
    uint32_t v[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (AWQ) {
        v[i] = fetch_code_awq(qw, kbase + off[i], n, size_n);
        v[4 + i] = fetch_code_awq(qw, kbase + off[i], n + 8, size_n);
      } else {
        v[i] = fetch_code(qw, perm, kbase + off[i], n, size_n);
        v[4 + i] = fetch_code(qw, perm, kbase + off[i], n + 8, size_n);
      }
    }
    out[idx] = interleave_pack(v);
  }
}

// 8-bit codes, native layout: one thread per output word of one nibble plane.
__global__ __launch_bounds__(256) void repack_native8_kernel(const uint32_t* __restrict__ qw,
                                                              const int32_t* __restrict__ perm,
                                                              uint32_t* __restrict__ out, int64_t size_k,
                                                              int64_t size_n) {
  const int64_t total = size_k * size_n / 4;
  const int64_t k_tiles = size_k / 128;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int j = idx & 3;
    const int lane = (idx >> 2) & 63;
    const int plane = (idx >> 8) & 1;
    const int64_t tile = idx >> 9;
    const int64_t nt = tile / k_tiles, kt = tile - nt * k_tiles;
    const int o = lane >> 4, r = lane & 15;
    const int64_t k0 = kt * 128 + j * 32 + o * 8;
    const int64_t n = nt * 16 + r;
    uint32_t v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint32_t c = fetch_code8(qw, perm, k0 + e, n, size_n);
      v[e] = plane ? (c & 0xFu) : (c >> 4);
    }
    out[idx] = interleave_pack(v);
  }
}

// 8-bit codes kept as bytes (NATIVE_BYTES): one thread per output word (four consecutive rows of one column).
__global__ __launch_bounds__(256) void repack_native8_bytes_kernel(const uint32_t* __restrict__ qw,
                                                                    const int32_t* __restrict__ perm,
                                                                    uint32_t* __restrict__ out, int64_t size_k,
                                                                    int64_t size_n) {
  const int64_t total = size_k * size_n / 4;
  const int64_t k_tiles = size_k / 128;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int q = idx & 3;
    const int lane = (idx >> 2) & 63;
    const int h = (idx >> 8) & 1;
    const int64_t tile = idx >> 9;
    const int64_t nt = tile / k_tiles, kt = tile - nt * k_tiles;
    const int o = lane >> 4, r = lane & 15;
    const int j = 2 * h + (q >> 1);
    const int64_t k0 = kt * 128 + j * 32 + o * 8 + (q & 1) * 4;
    const int64_t n = nt * 16 + r;
    uint32_t res = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) res |= fetch_code8(qw, perm, k0 + e, n, size_n) << (8 * e);
    out[idx] = res;
  }
}

// 8-bit codes, reference (Marlin) order: one thread per output word.
__global__ __launch_bounds__(256) void repack_marlin8_kernel(const uint32_t* __restrict__ qw,
                                                              const int32_t* __restrict__ perm,
                                                              uint32_t* __restrict__ out, int64_t size_k,
                                                              int64_t size_n) {
  const int64_t total = size_k * size_n / 4;
  const int64_t n_tiles = size_n / 64;
  for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
       idx += (int64_t)gridDim.x * blockDim.x) {
    const int which = idx & 1;
    const int warp = (idx >> 1) & 3;
    const int th = (idx >> 3) & 31;
    const int64_t tile = idx >> 8;
    const int64_t kt = tile / n_tiles, nt = tile - kt * n_tiles;
    const int64_t n = nt * 64 + warp * 16 + (th >> 2) + which * 8;
    const int64_t kbase = kt * 16 + (th & 3) * 2;
    const int off[4] = {0, 8, 1, 9};     // byte i <- row offset {0, 1, 8, 9}[{0, 2, 1, 3}[i]]
    uint32_t res = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) res |= fetch_code8(qw, perm, kbase + off[i], n, size_n) << (8 * i);
    out[idx] = res;
  }
}

// ----------------------------------------------------------------------------- native order, whole tiles
// The three kernels below write every output tile as the 16-byte pieces its lanes own (a wavefront store is contiguous)
// and read the checkpoint tensor in whole 64-byte pieces or more.  Bound: HBM.  What the one-word-per-thread kernels above
// lose is the gather: 8 four-byte loads per output word with act_order or AWQ, from lines that other workgroups fetch again.
// They stay for the MARLIN order, for pointers that are not 16-byte aligned, and for act_order on long narrow layers (strips beyond
// LDS, or too few of them).

// OUT 0: 4-bit codes; 1: 8-bit codes as two nibble planes; 2: 8-bit codes as bytes.
template <int OUT>
__device__ inline void put_code(v4u& lo, v4u& hi, int j, int e, uint32_t word, int shift) {
  constexpr int pos[8] = {0, 4, 1, 5, 2, 6, 3, 7};      // nibble position of element e
  if constexpr (OUT == 0) {
    lo[j] |= ((word >> shift) & 0xFu) << (4 * pos[e]);
  } else if constexpr (OUT == 1) {
    const uint32_t b = word >> shift;
    lo[j] |= ((b >> 4) & 0xFu) << (4 * pos[e]);      // plane 0: high nibbles
    hi[j] |= (b & 0xFu) << (4 * pos[e]);
  } else {      // lane's 16 bytes of block h = j / 2: word 2 (j & 1) + e / 4, byte e % 4
    const uint32_t b = ((word >> shift) & 0xFFu) << (8 * (e & 3));
    if (j < 2) lo[2 * (j & 1) + (e >> 2)] |= b;
    else hi[2 * (j & 1) + (e >> 2)] |= b;
  }
}

template <int OUT>
__device__ inline void store_tile(uint32_t* __restrict__ out, int64_t tile, int lane, const v4u& lo, const v4u& hi) {
  v4u* o = reinterpret_cast<v4u*>(out);
  if constexpr (OUT == 0) {
    o[tile * 64 + lane] = lo;
  } else {
    o[tile * 128 + lane] = lo;
    o[tile * 128 + 64 + lane] = hi;
  }
}

constexpr int64_t REPACK_LDS_MAX = 160 * 1024;
// act_order: output row k takes input row perm[k], anywhere in K.  A workgroup holds one strip of 4 C columns of the whole
// checkpoint tensor in LDS (K / 8 rows of 16 C bytes; 8-bit: K / 4) and gathers from there.  A thread builds the pieces of C
// lanes (o, r = 4c + q for c = 0 .. C - 1), so that an index is looked up and turned into an address and a shift once for
// C columns, which one LDS read brings: the strip is kept column-transposed (position C q + c holds column
// 4c + q), and the four lanes q of one store are neighbours.  Strips that share a 128-byte line run on one XCD.  A thread's
// first 32 indexes are requested ahead of the barrier: their round trip is over when the strip has arrived.
// Measured, us, indexes behind the barrier -> this: 4096 x 28672 (4 bits, 117 MB in and out) 29.6 -> 28.8 = 4.1 TB/s, 8192 x 8192
// 20.2 -> 18.9, 4096 x 4096 7.6 -> 6.9; the random rows cost LDS bank conflicts, so that it stays behind the 20 us of the kernel
// without a permutation.  Two, four or eight loads of the strip in flight per thread instead of one: 0 .. 10 % slower.
template <int OUT, int C>
__global__ __launch_bounds__(1024, 6) void repack_native_perm_kernel(const uint32_t* __restrict__ qw, const int32_t* __restrict__ perm,
                                                                     uint32_t* __restrict__ out, int size_k, int size_n,
                                                                     int strips_per_xcd) {
  static_assert(C == 2 || C == 4, "half or whole tiles");
  extern __shared__ __attribute__((aligned(16))) uint32_t strip[];
  typedef uint32_t Row __attribute__((ext_vector_type(C)));
  const int st = (int)(blockIdx.x & 7) * strips_per_xcd + (int)(blockIdx.x >> 3);
  if (st * 4 * C >= size_n) return;
  constexpr int LOG_ROWS = OUT == 0 ? 3 : 2;      // codes per word, log2
  const int k_tiles = size_k >> 7, pieces = k_tiles * 16;
  const v4i* order = reinterpret_cast<const v4i*>(perm);
  v4i idx[8];
  auto request = [&](int i) {      // the 32 indexes of piece i: rows 32 j + 8 o + e of its tile
#pragma unroll
    for (int j = 0; j < 8; ++j) idx[j] = order[(i >> 4) * 32 + (j >> 1) * 8 + ((i >> 2) & 3) * 2 + (j & 1)];
  };
  const int chunks = (size_k >> LOG_ROWS) * C;
  for (int i = threadIdx.x; i < chunks; i += blockDim.x) {
    const int row = i / C, c = i % C;
    const v4u w = *reinterpret_cast<const v4u*>(qw + (int64_t)row * size_n + st * 4 * C + 4 * c);
#pragma unroll
    for (int q = 0; q < 4; ++q) strip[row * 4 * C + C * q + c] = w[q];
  }
  if ((int)threadIdx.x < pieces) request(threadIdx.x);
  __syncthreads();
  for (int i = threadIdx.x; i < pieces; i += blockDim.x) {
    const int q = i & 3, o = (i >> 2) & 3, kt = i >> 4;
    v4u lo[C] = {}, hi[C] = {};
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int src = idx[2 * j + (e >> 2)][e & 3];
        const Row w = *reinterpret_cast<const Row*>(strip + (src >> LOG_ROWS) * 4 * C + C * q);
        const int shift = (src & ((1 << LOG_ROWS) - 1)) * (32 >> LOG_ROWS);
#pragma unroll
        for (int c = 0; c < C; ++c) put_code<OUT>(lo[c], hi[c], j, e, w[c], shift);
      }
    const int64_t tile = (int64_t)(st * C / 4) * k_tiles + kt;
#pragma unroll
    for (int c = 0; c < C; ++c) store_tile<OUT>(out, tile, 16 * o + 4 * (st * C % 4 + c) + q, lo[c], hi[c]);
    if (i + (int)blockDim.x < pieces) request(i + blockDim.x);
  }
}

// GPTQ order kept: a lane's 8 codes of one word are one input word (8-bit: two).  A wavefront makes one tile, the four of
// a workgroup neighbouring tiles of one K step (256 contiguous bytes per input row).  4096 x 28672: 20.3 us = 5.8 TB/s.
template <int OUT>
__global__ __launch_bounds__(256) void repack_native_rows_kernel(const uint32_t* __restrict__ qw, uint32_t* __restrict__ out, int size_k,
                                                                 int size_n) {
  const int lane = threadIdx.x & 63, o = lane >> 4, r = lane & 15;
  const int nt = blockIdx.x * 4 + (threadIdx.x >> 6), kt = blockIdx.y;
  const uint32_t* src = qw + nt * 16 + r;
  v4u lo = {}, hi = {};
  uint32_t w[4][OUT == 0 ? 1 : 2];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int64_t octet = (int64_t)kt * 16 + j * 4 + o;
    if constexpr (OUT == 0) {
      w[j][0] = src[octet * size_n];
    } else {
      w[j][0] = src[octet * 2 * size_n];
      w[j][1] = src[(octet * 2 + 1) * size_n];
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int e = 0; e < 8; ++e)
      put_code<OUT>(lo, hi, j, e, OUT == 0 ? w[j][0] : w[j][e >> 2], OUT == 0 ? 4 * e : 8 * (e & 3));
  store_tile<OUT>(out, (int64_t)nt * (size_k >> 7) + kt, lane, lo, hi);
}

// AWQ: input rows are K, a word holds 8 columns of one row.  A workgroup takes 128 rows x 256 columns (whole 128-byte lines;
// 64 columns per workgroup: 45.9 us) through LDS; a lane's output word is 8 rows' nibbles of its column.  4096 x 28672:
// 23.4 us = 5.0 TB/s.
__global__ __launch_bounds__(256) void repack_native_awq_kernel(const uint32_t* __restrict__ qw, uint32_t* __restrict__ out, int size_k,
                                                                int size_n) {
  constexpr int PITCH = 33;      // words per row: the rows of one o and of the next start in different banks
  __shared__ uint32_t tile_in[128 * PITCH];
  const int kt = blockIdx.y, n_words = size_n >> 3, w0 = blockIdx.x * 32;
  const int words = n_words - w0 < 32 ? n_words - w0 : 32;      // (a multiple of 8)
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = i * 32 + (threadIdx.x >> 3), c = (threadIdx.x & 7) * 4;
    if (c < words) {
      const v4u w = *reinterpret_cast<const v4u*>(qw + ((int64_t)kt * 128 + row) * n_words + w0 + c);
#pragma unroll
      for (int q = 0; q < 4; ++q) tile_in[row * PITCH + c + q] = w[q];
    }
  }
  __syncthreads();
  const int lane = threadIdx.x & 63, o = lane >> 4, r = lane & 15;
  const int shift = (((r & 1) << 2) | ((r & 7) >> 1)) * 4;
  for (int t = threadIdx.x >> 6; 2 * t < words; t += 4) {
    v4u lo = {}, hi = {};
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 8; ++e) put_code<0>(lo, hi, j, e, tile_in[(j * 32 + o * 8 + e) * PITCH + t * 2 + (r >> 3)], shift);
    store_tile<0>(out, (int64_t)(blockIdx.x * 16 + t) * (size_k >> 7) + kt, lane, lo, hi);
  }
}

// Whether the kernels above take a problem: 16-byte pointers, 32-bit indexes, and with act_order a strip that fits LDS.  Where only
// strips of 8 columns fit, a layer has to be wide enough to give work to many compute units: a strip takes 10 .. 25 us by
// itself, and up to these widths the kernels of one word per thread are ahead or within a few percent (K = 24064 x 64 columns, 4 bits, 12.0
// against 5.1 us, 25600 x 512 19.7 against 18.8, x 640 18.9 against 21.5; 8 bits 17920 x 384 21.2 against 20.7, x 448 20.2 against 22.7;
// bytes 17920 x 768 24.2 against 22.6, x 896 18.0 against 22.3).
static bool repack_tiles_ok(const void* qweight, const void* perm, const void* out, int64_t size_k, int64_t size_n, int num_bits, int layout) {
  if (((uintptr_t)qweight % 16) || ((uintptr_t)out % 16) || ((uintptr_t)perm % 16)) return false;
  if (size_k > (1 << 22) || size_n > (1 << 24)) return false;
  if (!perm || size_k * num_bits * 2 <= REPACK_LDS_MAX) return true;
  return size_k * num_bits <= REPACK_LDS_MAX && size_n > (num_bits == 4 ? 512 : layout == VAQ_LAYOUT_NATIVE ? 384 : 768);
}

template <int OUT, int C>
static int launch_repack_perm(const uint32_t* qw, const int32_t* perm, uint32_t* out, int64_t size_k, int64_t size_n, hipStream_t s) {
  const size_t lds = (size_t)size_k * C * (OUT == 0 ? 2 : 4);
  static size_t reserved[VAQ_MAX_DEVICES];
  const int rc = reserve_dynamic_lds(reinterpret_cast<const void*>(&repack_native_perm_kernel<OUT, C>), lds, reserved, "w4a16_repack");
  if (rc != VAQ_OK) return rc;
  const int per_xcd = (int)((size_n / (4 * C) + 7) / 8);
  // 12 wavefronts: 8 are up to 12 % slower where a compute unit holds one strip (8 bits 8192 x 8192 39.6 against 34.5 us), 16 up to 6 %
  // where it holds two (4096 x 28672 29.8 against 28.2).  Single whole strips of nibbles take 16 (14336 x 4096 17.6 -> 17.2), of 8 bits
  // where there are more of them than compute units (8192 x 14336 70.2 -> 68.6, 6144 x 28672 100.5 -> 96.4; 8192 x 4096 18.3 against
  // 18.7).  A whole strip of few 16-byte loads takes no more threads than loads: more of them share a compute unit (128 x 14336 6.4 ->
  // 4.7 us in 8 bits, 4.6 -> 3.5 in 4; 512 x 28672 7.7 -> 7.0 in 4 bits, 11.4 -> 10.9 in 8; 384 x 16192 7.8 -> 6.7 in 8).
  // And three workgroups of 8 wavefronts where they hold all strips at once and two of 12 do not (2560 x 8384 in 8 bits 18.5 -> 16.0).
  const int64_t loads = size_k / (OUT == 0 ? 8 : 4) * C, strips = size_n / (4 * C), cus = num_cus_current_device();
  const bool single = lds > REPACK_LDS_MAX / 2 && OUT != 2 && (OUT == 0 || strips > cus);
  const bool three = lds > REPACK_LDS_MAX / 5 && lds * 3 <= REPACK_LDS_MAX && strips > 2 * cus && strips <= 3 * cus;
  const int threads = C != 4 ? 768 : loads <= 512 ? (loads <= 256 ? 256 : (int)(loads + 63) / 64 * 64) : three ? 512 : single ? 1024 : 768;
  hipLaunchKernelGGL((repack_native_perm_kernel<OUT, C>), dim3(per_xcd * 8), dim3(threads), lds, s, qw, perm, out, (int)size_k, (int)size_n,
                     per_xcd);
  return VAQ_OK;
}

template <int OUT>
static int launch_repack_tiles(const uint32_t* qw, const int32_t* perm, uint32_t* out, int64_t size_k, int64_t size_n, hipStream_t s) {
  if (!perm) {
    hipLaunchKernelGGL(repack_native_rows_kernel<OUT>, dim3((unsigned)(size_n / 64), (unsigned)(size_k / 128)), dim3(256), 0, s, qw, out,
                       (int)size_k, (int)size_n);
    return VAQ_OK;
  }
  // Strips of 16 columns read and write whole 64-byte pieces and look an index up once for four columns.  Strips of 8 take K up to
  // twice as far (one word per thread beyond: 8 bits 14336 x 4096 137 -> 40 us, 4 bits 24576 x 2048 58 -> 21), and
  // give every compute unit one where 16 columns leave half of them idle (5120 x 1024 6.0 -> 4.8 us); with as many strips as
  // compute units they are the slower ones (4096 x 4096 6.9 against 8.0 us).
  const bool half = size_k * (OUT == 0 ? 8 : 16) > REPACK_LDS_MAX || size_n / 8 <= num_cus_current_device();
  return half ? launch_repack_perm<OUT, 2>(qw, perm, out, size_k, size_n, s) : launch_repack_perm<OUT, 4>(qw, perm, out, size_k, size_n, s);
}

}  // namespace vaq

static int repack_common(const int32_t* qweight, const int32_t* perm, int32_t* out, int64_t size_k, int64_t size_n,
                         int num_bits, int layout, bool awq, void* stream) {
  using namespace vaq;
  VAQ_CHECK_ARG(num_bits == 4 || num_bits == 8, "w4a16_repack: num_bits must be 4 or 8. Got = %d", num_bits);
  VAQ_CHECK_SUPPORTED(num_bits == 4 || !awq, "w4a16_repack: 8-bit AWQ weights are not built");
  VAQ_CHECK_ARG(size_k > 0 && size_k % 16 == 0, "w4a16_repack: size_k = %lld is not divisible by tile_k_size = 16",
                (long long)size_k);
  VAQ_CHECK_ARG(size_n > 0 && size_n % 64 == 0, "w4a16_repack: size_n = %lld is not divisible by tile_n_size = 64",
                (long long)size_n);
  VAQ_CHECK_ARG(layout == VAQ_LAYOUT_MARLIN || layout == VAQ_LAYOUT_NATIVE || layout == VAQ_LAYOUT_NATIVE_BYTES,
                "w4a16_repack: unknown layout %d", layout);
  VAQ_CHECK_ARG(layout != VAQ_LAYOUT_NATIVE_BYTES || (num_bits == 8 && !awq),
                "w4a16_repack: the byte layout is for 8-bit GPTQ-packed weights");
  VAQ_CHECK_ARG(layout == VAQ_LAYOUT_MARLIN || size_k % 128 == 0,
                "w4a16_repack: native layout needs size_k %% 128 == 0, got size_k = %lld", (long long)size_k);
  VAQ_CHECK_ARG(qweight && out, "w4a16_repack: null pointer");
  const int64_t total = size_k * size_n / (32 / num_bits);
  const int threads = 256;
  int64_t blocks = (total + threads - 1) / threads;
  const int64_t cap = (int64_t)num_cus_current_device() * 16;
  if (blocks > cap) blocks = cap;
  hipStream_t s = (hipStream_t)stream;
  const uint32_t* qw = (const uint32_t*)qweight;
  uint32_t* o = (uint32_t*)out;
  const dim3 grid((unsigned)blocks), block(threads);
  if (layout != VAQ_LAYOUT_MARLIN && repack_tiles_ok(qweight, perm, out, size_k, size_n, num_bits, layout)) {
    int rc = VAQ_OK;
    if (awq)
      hipLaunchKernelGGL(repack_native_awq_kernel, dim3((unsigned)((size_n + 255) / 256), (unsigned)(size_k / 128)), dim3(256), 0, s, qw, o,
                         (int)size_k, (int)size_n);
    else if (num_bits == 4) rc = launch_repack_tiles<0>(qw, perm, o, size_k, size_n, s);
    else if (layout == VAQ_LAYOUT_NATIVE) rc = launch_repack_tiles<1>(qw, perm, o, size_k, size_n, s);
    else rc = launch_repack_tiles<2>(qw, perm, o, size_k, size_n, s);
    if (rc != VAQ_OK) return rc;
  } else if (num_bits == 8) {
    if (layout == VAQ_LAYOUT_NATIVE) hipLaunchKernelGGL(repack_native8_kernel, grid, block, 0, s, qw, perm, o, size_k, size_n);
    else if (layout == VAQ_LAYOUT_NATIVE_BYTES) hipLaunchKernelGGL(repack_native8_bytes_kernel, grid, block, 0, s, qw, perm, o, size_k, size_n);
    else hipLaunchKernelGGL(repack_marlin8_kernel, grid, block, 0, s, qw, perm, o, size_k, size_n);
  } else if (layout == VAQ_LAYOUT_NATIVE) {
    if (awq)
      hipLaunchKernelGGL((repack_native_kernel<false, true>), grid, block, 0, s, qw, perm, o, size_k, size_n);
    else if (perm)
      hipLaunchKernelGGL((repack_native_kernel<true, false>), grid, block, 0, s, qw, perm, o, size_k, size_n);
    else
      hipLaunchKernelGGL((repack_native_kernel<false, false>), grid, block, 0, s, qw, perm, o, size_k, size_n);
  } else {
    if (awq)
      hipLaunchKernelGGL(repack_marlin_kernel<true>, grid, block, 0, s, qw, perm, o, size_k, size_n);
    else
      hipLaunchKernelGGL(repack_marlin_kernel<false>, grid, block, 0, s, qw, perm, o, size_k, size_n);
  }
  VAQ_CHECK_LAUNCH("w4a16_repack");
  return VAQ_OK;
}

extern "C" int vaq_w4a16_repack(const int32_t* qweight, const int32_t* perm, int32_t* out, int64_t size_k,
                                int64_t size_n, int num_bits, int layout, void* stream) {
  return repack_common(qweight, perm, out, size_k, size_n, num_bits, layout, false, stream);
}

extern "C" int vaq_w4a16_repack_awq(const int32_t* qweight, int32_t* out, int64_t size_k, int64_t size_n, int num_bits,
                                    int layout, void* stream) {
  return repack_common(qweight, nullptr, out, size_k, size_n, num_bits, layout, true, stream);
}
