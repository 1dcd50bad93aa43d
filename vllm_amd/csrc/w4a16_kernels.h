// The kernels behind the W4A16 GEMM, as its entry point (w4a16_gemm.hip) sees them.
#pragma once
#include "vaq_common.h"

namespace vaq {
// `sub` = quantisation groups per 128-row weight tile (1, 2, 4); `channelwise` = one scale row for all of K (sub == 1)
int w4a16_decode_workspace(int M, int N, int K, size_t* c_tmp_bytes, size_t* counter_ints);
int w4a16_decode_launch(const void* a, int64_t lda, const int32_t* b, const void* scales, const int32_t* zeros,
                        const int32_t* perm, const void* bias, void* c, float* c_tmp, int64_t c_tmp_bytes,
                        int32_t* counters, int64_t counter_ints, int M, int N, int K, bool channelwise, int dtype,
                        hipStream_t s);
int w4a16_decode2_workspace(int M, int N, int K, int sub, bool w8, size_t* c_tmp_bytes, size_t* counter_ints);
// Which kernel takes more than 16 rows: the tile kernel, the decode kernel's workgroups of all rows, or of 16 rows each.
enum { D2_TILE, D2_WORKGROUP, D2_ROWS };
int w4a16_decode2_choose(int M, int N, int K, int sub, int wt, bool act_order, bool has_perm, bool wg_ok, bool tile_ok, double tile_us);
// What the choice of a tile depends on: 4-bit codes in groups of 128 rows / channelwise, in smaller groups, 8-bit codes likewise and in groups
// of 32, FP8 weights (and two to price calls by: plain codes on the shapes with weights through LDS only, smaller groups on what the kernel with activations in registers is weighed against).
enum TileFormat { TILES_PLAIN, TILES_SUB, TILES_8BIT, TILES_8BIT_64, TILES_8BIT_32, TILES_FP8, TILES_PLAIN_STAGED, TILES_SUB_WEIGHED };
inline TileFormat tile_format(int sub, int wt) {
  if (wt == 1) return sub == 1 ? TILES_8BIT : sub == 2 ? TILES_8BIT_64 : TILES_8BIT_32;
  return wt == 2 ? TILES_FP8 : sub > 1 ? TILES_SUB : TILES_PLAIN;
}
double w4a16_decode2_us(int M, int N, int K, int sub, bool w8, bool rows);      // predicted time of the decode kernel's plan
double w4a16_decode2_gather_us(int M, int N, int K, int sub, bool w8, double* gather);      // with act_order gathered inside it; `gather`: its share
double w4a16_staged_us(int M, int N, int K, bool plain);
double w4a16_tile_us(int M, int N, int K, TileFormat format);
int w4a16_decode2_launch(const void* a, int64_t lda, const int32_t* b, const void* scales, const int32_t* zeros,
                         const int32_t* perm, const void* bias, void* c, float* c_tmp, int64_t c_tmp_bytes,
                         int32_t* counters, int64_t counter_ints, int M, int N, int K, int sub, bool channelwise,
                         int wt, int dtype, bool rows, hipStream_t s);      // wt: 0 4-bit codes, 1 8-bit codes, 2 FP8 e4m3 bytes
// The kernel with activations in registers (w4a16_regs.hip), up to REGS_MAX_M rows, no act_order, no FP8 weights: predicted time (negative: it
// does not take the problem), scratch, launch.
constexpr int REGS_MAX_M = 256;
double w4a16_regs_us(int M, int N, int K, int sub, int wt, int* n_tiles = nullptr, int* wavefronts = nullptr);      // ... of its plan
bool w4a16_takes_regs(int M, int N, int K, int sub, int wt, double* other, bool act_order = false);      // w4a16_gemm.hip; *other: predicted time of what takes it otherwise
void w4a16_regs_workspace(int M, int N, int K, int sub, bool w8, size_t* c_tmp_bytes, size_t* counter_ints);
int w4a16_regs_launch(const void* a, int64_t lda, const int32_t* b, const void* scales, const int32_t* zeros, const void* bias, void* c,
                      float* c_tmp, int32_t* counters, int M, int N, int K, int sub, bool channelwise, bool w8, int dtype, hipStream_t s);
int w4a16_prefill_workspace(int M, int N, int K, TileFormat format, size_t* c_tmp_bytes, size_t* counter_ints);
int w4a16_prefill_launch(const void* a, int64_t lda, const int32_t* b, const void* scales, const int32_t* zeros,
                         const void* bias, void* c, float* c_tmp, int64_t c_tmp_bytes, int32_t* counters,
                         int64_t counter_ints, int M, int N, int K, int sub, bool channelwise, int wt, int dtype,
                         hipStream_t s);

}  // namespace vaq
