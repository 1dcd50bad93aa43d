/*
 * vaq_tuning.h -- kernel-variant overrides for this library's own tests and benchmarks.  Not part of the drop-in
 * surface (include/vllm_amd_qlinear.h): the reference's kernels take no such argument and the ops never pass one.
 * The struct layout is mirrored by vllm_amd/_lib.py and may change with the kernels.
 */
#ifndef VAQ_TUNING_H_
#define VAQ_TUNING_H_

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif
#pragma GCC visibility push(default)

/*
 * Kernel-variant overrides for tests and benchmarks.  No counterpart in the reference (its kernels take no such
 * argument); the drop-in surface never passes one.  A VaqTuning applies to the ONE call it is handed to, on the calling
 * thread only: the library keeps no tuning state between calls.  Every field: 0 = the automatic choice.
 */
typedef struct VaqTuning {
  int decode_impl;      /* W4A16 decode kernel: 1 LDS-staged activations, 2 register-resident activations          */
  int decode2_gs;       /* LDS-staged kernel: weight tiles per wavefront                                             */
  int decode2_wks;      /*   K slices per workgroup                                                                  */
  int decode2_wn;       /*   n-tiles per workgroup                                                                   */
  int decode_tg;        /* register-resident kernel: groups per wavefront                                            */
  int decode_wk;        /*   wavefronts along K per workgroup                                                        */
  int decode_gx;        /*   workgroups along N                                                                      */
  int decode_depth;     /*   prefetch depth                                                                          */
  int prefill_tile;     /* W4A16 tile kernel: tile id + 1                                                            */
  int prefill_split;    /*   K split                                                                                 */
  int fp8_path;         /* FP8 GEMM: 1 weight-streaming kernel, 2 tile kernel                                        */
  int fp8_tile_impl;    /*   1 register-staged tile kernel                                                           */
  int fp8_tile_cfg;     /*   multi-stage tile shape id, -1 = two-stage kernel                                        */
  int fp8_split;        /*   K split of the tile kernel                                                              */
  int fp8_gx;           /*   workgroups of the weight-streaming kernel                                               */
  int fp8_stream_split; /*   -1 = never run the weight-streaming kernel over two halves of K                         */
  int quant_wg_per_row; /* per-token FP8 quant: 1 = one workgroup per row, 2 = one wavefront per row (where it can)    */
  int exp[15];          /* further switches of the same kind, for A/B timing runs: [0] = 1 shared instead of private  */
                        /*   activation fill, [1] = ring variant + 1, [2] rows over workgroups (1 off, 2 forced) of   */
                        /*   the LDS-staged decode kernel, [3] = 1 sixteen staged rows for M = 5 .. 8, [5] = 1 two K   */
                        /*   slabs never merged into one; [4] FP8 streaming through LDS (1 / 2 / 3 = 8 / 4 / 16 steps   */
                        /*   per wavefront, 9 = off); [10] = 1 both tile kernels: never split only the tiles of a half-empty last round; */
                        /*   [12] = 1 FP8 tile kernel: every tile starts at the first K step; [13] = 1 FP8 tile kernel: no tile  */
                        /*   row past M; [14] > 0 W4A16 tile kernel: KiB that the partial tiles of a K split may take; [6] > 1 both tile     */
                        /*   kernels, 256 x 256 tiles: the tiles of the last round in this many parts of K; [9] = 1 act_order: columns */
                        /*   permuted by a launch of its own for the W4A16 tile kernel only; [11] FP8 kernel for some dozen rows: 1 never, else */
                        /*   its plan, n-tiles | m-blocks << 4;                                                                      */
                        /*   [8] W4A16 kernel with activations in registers: 1 never, else its plan, n-tiles | m-blocks << 4 |        */
                        /*   wavefronts << 8 | parts of K << 12;                                                                     */
                        /*   [7] = 1 LDS-staged decode kernel: n-tiles in launch order, not grouped by XCD             */
} VaqTuning;

/* The entry points of the same name without `_tuned`, with `tuning` (may be NULL) applied to this call. */
int vaq_w4a16_gemm_workspace_tuned(int64_t size_m, int64_t size_n, int64_t size_k, int has_perm, int device,
                                   size_t* c_tmp_bytes, size_t* a_tmp_bytes, size_t* counter_ints,
                                   const VaqTuning* tuning);
int vaq_w4a16_gemm_tuned(const void* a, int64_t lda, const int32_t* b, const void* scales, const int32_t* zeros,
                         const int32_t* perm, const void* bias, void* c, float* c_tmp, int64_t c_tmp_bytes, void* a_tmp,
                         int32_t* counters, int64_t counter_ints, int64_t size_m, int64_t size_n, int64_t size_k,
                         int group_size, int dtype, int wtype, int force_path, void* stream, const VaqTuning* tuning);
int vaq_fp8_scaled_mm_workspace_tuned(int64_t size_m, int64_t size_n, int64_t size_k, size_t* c_tmp_bytes,
                                      size_t* counter_ints, const VaqTuning* tuning);
int vaq_fp8_scaled_mm_ws_tuned(const uint8_t* a, int64_t lda, const uint8_t* b, int64_t ldb, const float* sa,
                               int64_t sa_count, const float* sb, int64_t sb_count, const void* bias, void* out,
                               int64_t ldc, int out_dtype, int64_t size_m, int64_t size_n, int64_t size_k, float* c_tmp,
                               int64_t c_tmp_bytes, int32_t* counters, int64_t counter_ints, void* stream,
                               const VaqTuning* tuning);
int vaq_fp8_quant_per_token_tuned(const void* in, int in_dtype, int64_t in_row_stride, uint8_t* out,
                                  int64_t out_row_stride, float* scales, const float* scale_ub, int64_t rows,
                                  int64_t hidden, void* stream, const VaqTuning* tuning);

/*
 * The plan of the W4A16 decode kernel for a problem, without launching anything: plan[0 .. 5] = weight tiles per wavefront, K
 * slices and n-tiles per workgroup, parts of K, staged rows, predicted us (negative: no plan).  `sub` = groups per 128
 * rows, `w8` = 8-bit codes, `kind` = 0 workgroups of all rows, 1 the same by the rule instead of the price, 2 of 16 rows.
 */
int vaq_w4a16_decode_plan(int64_t size_m, int64_t size_n, int64_t size_k, int sub, int w8, int kind, double* plan);

/*
 * The same of the W4A16 kernel with activations in registers: plan[0 .. 6] = n-tiles, m-blocks and wavefronts of a workgroup, parts of K,
 * predicted us, predicted us of the kernel that takes the problem otherwise, 1 if this one takes it.
 */
int vaq_w4a16_regs_plan(int64_t size_m, int64_t size_n, int64_t size_k, int sub, int w8, double* plan);

/* The same of the FP8 kernel for some dozen rows: plan[0 .. 4] = n-tiles, m-blocks, predicted us, us of what takes it otherwise, 1 if it takes it. */
int vaq_fp8_regs_plan(int64_t size_m, int64_t size_n, int64_t size_k, double* plan);

/*
 * The same of the W4A16 tile kernels: plan[0 .. 3] = tile id (48: the 256 x 256 kernel of w4a16_tile256_kernel.h, others from 41 on: strips), parts of K,
 * first tile that is split where only those of the last round are (else 0), predicted us.  `wt` = 0 4-bit, 1 8-bit codes, 2 FP8 weights; `staged` = 1: the cheapest plan
 * of the shapes with weights through LDS, whose price the decode kernels are weighed against.
 */
int vaq_w4a16_tile_plan(int64_t size_m, int64_t size_n, int64_t size_k, int sub, int wt, int staged, double* plan);

#pragma GCC visibility pop
#ifdef __cplusplus
}
#endif
#endif /* VAQ_TUNING_H_ */
