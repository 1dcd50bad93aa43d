// out[m, k] = a[m, perm[k]] for 16-bit elements (activation reorder for act_order weights).
#include "vaq_common.h"

namespace vaq {

// One workgroup per row; each thread gathers 8 columns and writes them as one 16-byte store.
__global__ __launch_bounds__(256) void permute_cols_kernel(const uint16_t* __restrict__ a, int64_t lda,
                                                            const int32_t* __restrict__ perm,
                                                            uint16_t* __restrict__ out, int64_t size_k) {
  const int64_t m = blockIdx.x;
  const uint16_t* row = a + m * lda;
  uint16_t* orow = out + m * size_k;
  const int64_t chunks = size_k / 8;
  for (int64_t c = threadIdx.x; c < chunks; c += blockDim.x) {
    const v4i p0 = *reinterpret_cast<const v4i*>(perm + c * 8);
    const v4i p1 = *reinterpret_cast<const v4i*>(perm + c * 8 + 4);
    v4u r;
    r.x = (uint32_t)row[p0.x] | ((uint32_t)row[p0.y] << 16);
    r.y = (uint32_t)row[p0.z] | ((uint32_t)row[p0.w] << 16);
    r.z = (uint32_t)row[p1.x] | ((uint32_t)row[p1.y] << 16);
    r.w = (uint32_t)row[p1.z] | ((uint32_t)row[p1.w] << 16);
    *reinterpret_cast<v4u*>(orow + c * 8) = r;
  }
}

// Rows staged in LDS: a workgroup copies PC_ROWS rows (as many as fit 32 KiB, so that several workgroups share a compute
// unit and one's loads overlap another's gathers) with coalesced 16-byte loads, then every thread gathers 8 columns
// per row from LDS (the permutation entries are read once and reused for all the rows) and writes 16-byte stores.
// The scattered 2-byte reads thus hit LDS instead of going out as 64 separate addresses per global load instruction.
// What bounds hundreds of rows is the chain of load, barrier, gather and store in each workgroup, so the first permutation
// entries are requested together with the rows, and few rows are dealt out one to a workgroup (see the launch).
template <int PC_ROWS>
__global__ __launch_bounds__(512) void permute_cols_lds_kernel(const uint16_t* __restrict__ a, int64_t lda,
                                                                const int32_t* __restrict__ perm,
                                                                uint16_t* __restrict__ out, int64_t size_m, int size_k) {
  extern __shared__ __attribute__((aligned(16))) uint16_t rows[];      // [PC_ROWS][size_k]
  const int64_t m0 = (int64_t)blockIdx.x * PC_ROWS;
  const int chunks = size_k / 8, threads = blockDim.x;
  const bool aligned = (lda % 8 == 0) && ((reinterpret_cast<uintptr_t>(a) & 15) == 0);
  const int c0 = min((int)threadIdx.x, chunks - 1);
  v4i p0 = *reinterpret_cast<const v4i*>(perm + c0 * 8), p1 = *reinterpret_cast<const v4i*>(perm + c0 * 8 + 4);
#pragma unroll
  for (int r = 0; r < PC_ROWS; ++r) {
    const int64_t m = m0 + r < size_m ? m0 + r : size_m - 1;
    const uint16_t* row = a + m * lda;
    if (aligned) {
      for (int c = threadIdx.x; c < chunks; c += threads)
        *reinterpret_cast<v4u*>(rows + (size_t)r * size_k + c * 8) = *reinterpret_cast<const v4u*>(row + c * 8);
    } else {
      for (int k = threadIdx.x; k < size_k; k += threads) rows[(size_t)r * size_k + k] = row[k];
    }
  }
  __syncthreads();
  for (int c = threadIdx.x; c < chunks;) {
#pragma unroll
    for (int r = 0; r < PC_ROWS; ++r) {
      if (m0 + r >= size_m) break;
      const uint16_t* row = rows + (size_t)r * size_k;
      v4u v;
      v.x = (uint32_t)row[p0.x] | ((uint32_t)row[p0.y] << 16);
      v.y = (uint32_t)row[p0.z] | ((uint32_t)row[p0.w] << 16);
      v.z = (uint32_t)row[p1.x] | ((uint32_t)row[p1.y] << 16);
      v.w = (uint32_t)row[p1.z] | ((uint32_t)row[p1.w] << 16);
      *reinterpret_cast<v4u*>(out + (m0 + r) * (int64_t)size_k + c * 8) = v;
    }
    c += threads;
    if (c < chunks) {
      p0 = *reinterpret_cast<const v4i*>(perm + c * 8);
      p1 = *reinterpret_cast<const v4i*>(perm + c * 8 + 4);
    }
  }
}

}  // namespace vaq

extern "C" int vaq_permute_cols(const void* a, int64_t lda, const int32_t* perm, void* out, int64_t size_m,
                                int64_t size_k, void* stream) {
  using namespace vaq;
  VAQ_CHECK_ARG(size_m >= 0 && size_k > 0, "permute_cols: bad shape [%lld, %lld]", (long long)size_m, (long long)size_k);
  VAQ_CHECK_ARG(size_k % 8 == 0, "permute_cols: size_k = %lld must be divisible by 8", (long long)size_k);
  VAQ_CHECK_ARG(lda >= size_k, "permute_cols: lda = %lld < size_k = %lld", (long long)lda, (long long)size_k);
  VAQ_CHECK_ARG(size_m < (1ll << 31), "permute_cols: size_m too large");
  if (size_m == 0) return VAQ_OK;
  VAQ_CHECK_ARG(a && perm && out, "permute_cols: null pointer");
  VAQ_CHECK_ARG(((uintptr_t)out % 16) == 0 && ((uintptr_t)perm % 16) == 0, "permute_cols: out/perm must be 16-byte aligned");
  const size_t row_bytes = (size_t)size_k * 2;
  if (row_bytes <= 128 * 1024) {
    // four or two rows to a workgroup only where that leaves two workgroups per compute unit: 4096 columns, 100 / 333 / 1024 rows
    // 4.0 / 4.2 / 5.0 -> 2.2 / 2.6 / 4.2 us (from one to the other, launch to launch), 4096 rows 12.3 us either way; and not from 1536
    // to 4095 columns, where one row is ahead at any number (2048 x 7500 16.1 -> 13.3 us, 3072 x 8192 26.0 -> 21.3, 1536 x 2048 5.9 ->
    // 4.6; 1024 x 8192 8.3 against 9.0 us, 4096 x 4096 13.1 against 14.9)
    const int64_t cus = num_cus_current_device(), few = 2 * cus;
    int rows = row_bytes * 4 <= 32 * 1024 ? 4 : (row_bytes * 2 <= 32 * 1024 ? 2 : 1);
    while (rows > 1 && (size_m / rows < few || (size_k >= 1536 && size_k < 4096))) rows /= 2;
    // One row: 512 threads for a long one (half the steps of the chain), four such workgroups to a compute unit.  More rows than that
    // run on 256 threads where all of them are on the device at once then (1280 x 12288 16.9 -> 14.9 us, 1280 x 14336 19.8 -> 18.0,
    // 1536 x 9088 15.0 -> 13.8), and shorter ones at any number (8192 x 3072 21.6 -> 21.3); else 512 are ahead again (4096 x 14336 54.2
    // against 48.7).
    const int64_t held = cus * (row_bytes * 8 < 160 * 1024 ? 8 : (160 * 1024 - 1) / (int64_t)row_bytes);
    const bool wide = rows == 1 && size_k > 2048 && (size_m <= 4 * cus || (size_m > held && size_k > 4096));
    const dim3 threads(wide ? 512 : 256);
    const size_t lds = rows * row_bytes;
    const void* kern = rows == 4 ? reinterpret_cast<const void*>(permute_cols_lds_kernel<4>)
                                 : (rows == 2 ? reinterpret_cast<const void*>(permute_cols_lds_kernel<2>)
                                              : reinterpret_cast<const void*>(permute_cols_lds_kernel<1>));
    if (lds > 64 * 1024 &&
        hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) {
      set_error("permute_cols: cannot reserve %zu bytes of LDS", lds);
      (void)hipGetLastError();
      return VAQ_ERR_LAUNCH;
    }
    const dim3 grid((unsigned)((size_m + rows - 1) / rows));
    if (rows == 4)
      hipLaunchKernelGGL(permute_cols_lds_kernel<4>, grid, threads, lds, (hipStream_t)stream, (const uint16_t*)a, lda, perm,
                         (uint16_t*)out, size_m, (int)size_k);
    else if (rows == 2)
      hipLaunchKernelGGL(permute_cols_lds_kernel<2>, grid, threads, lds, (hipStream_t)stream, (const uint16_t*)a, lda, perm,
                         (uint16_t*)out, size_m, (int)size_k);
    else
      hipLaunchKernelGGL(permute_cols_lds_kernel<1>, grid, threads, lds, (hipStream_t)stream, (const uint16_t*)a, lda, perm,
                         (uint16_t*)out, size_m, (int)size_k);
  } else {
    hipLaunchKernelGGL(permute_cols_kernel, dim3((unsigned)size_m), dim3(256), 0, (hipStream_t)stream,
                       (const uint16_t*)a, lda, perm, (uint16_t*)out, size_k);
  }
  VAQ_CHECK_LAUNCH("permute_cols");
  return VAQ_OK;
}
