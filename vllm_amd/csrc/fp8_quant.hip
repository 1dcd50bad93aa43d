// FP8 (OCP e4m3fn) activation quantisation for gfx950: per-token dynamic, per-tensor dynamic, per-tensor static.
//
// Bit-exactness contract (codes AND scales) with the reference kernels:
//   per token : amax = max|float(x)| ; s = max(min(amax, ub) / 448, 1/(448*512)) ; q = cvt(clamp(float(x) / s, +-448))
//               -- the correctly rounded fp32 quotient per element, not a reciprocal multiply (for 16-bit inputs without
//               an upper bound on the scale it comes from div16_exact: three instructions, the same bits);
//   per tensor: s = amax_all / 448 ; q = cvt(clamp(float(x) * (1 / s), +-448))   (reciprocal multiply);
//   static    : q = cvt(clamp(float(x) * (1 / scale), +-448)).
// cvt is the hardware v_cvt_pk_fp8_f32 (round-to-nearest-even; inputs are already clamped, NaN stays NaN).
// The file is compiled without fast-math, so `/` is the correctly rounded division.
//
// HBM-bound: each row is read ONCE -- a workgroup keeps its whole row in registers between the absmax pass and the
// convert pass whenever the row has at most 512 threads x 8 vectors x 8 elements = 32768 elements and its addresses and
// length allow vectors; other rows are read twice by single elements.  Per tensor, rows without gaps are one run of
// vectors, whatever their length.
#include "vaq_common.h"

namespace vaq {

constexpr float FP8_MAX = 448.0f;
// (measured: 512 threads with 4 vectors each against 256 x 8: 2.95 -> 2.68 us at 16 rows of 4096, 3.65 -> 3.3 us at 256
// rows, 41.5 -> 39.5 us at 4096 rows of 14336, unchanged at 4096 x 4096; 1024 x 2 and 128 x 16 are slower)
constexpr int QT = 512;         // threads per workgroup of the row-per-workgroup kernel (its TPB: QT or QT / 2)
constexpr int QTW = 256;        // threads per workgroup of the row-per-wavefront kernel (four rows)
constexpr int QTA = 1024;       // threads per workgroup of the maximum over a run

template <typename T>
__device__ inline float load_as_float(const T* p);
template <>
__device__ inline float load_as_float<float>(const float* p) { return *p; }
struct bf16_t { uint16_t v; };
struct f16_t { uint16_t v; };
template <>
__device__ inline float load_as_float<bf16_t>(const bf16_t* p) { return F16Traits<true>::to_float(p->v); }
template <>
__device__ inline float load_as_float<f16_t>(const f16_t* p) { return F16Traits<false>::to_float(p->v); }

__device__ inline float clamp448(float x) { return fmaxf(-FP8_MAX, fminf(x, FP8_MAX)); }

// two fp32 -> two e4m3fn codes in the low 16 bits
__device__ inline uint32_t cvt2(float a, float b) { return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(a, b, 0, false) & 0xffffu; }
__device__ inline uint8_t cvt1(float a) { return (uint8_t)(__builtin_amdgcn_cvt_pk_fp8_f32(a, a, 0, false) & 0xff); }

// 8 consecutive elements of a row: requested by load(), as floats after unpack().  Apart, because a conversion behind each load
// under its own condition waits for that load before the next is requested: four latencies for a row of 14336 instead of one.
template <typename T>
struct Vec8 {
  float f[8];
  v4u raw[sizeof(T) / 2];
  __device__ inline void load(const T* p) {
#pragma unroll
    for (int i = 0; i < (int)sizeof(T) / 2; ++i) raw[i] = reinterpret_cast<const v4u*>(p)[i];
  }
  __device__ inline void unpack() {
    const uint32_t* w = reinterpret_cast<const uint32_t*>(raw);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if constexpr (sizeof(T) == 2) {
        const T h{(uint16_t)(w[i / 2] >> (16 * (i & 1)))};
        f[i] = load_as_float<T>(&h);
      } else {
        f[i] = __builtin_bit_cast(float, w[i]);
      }
    }
  }
};

// MODE 0: dynamic per token (divide by row scale, scale written per row)
// MODE 1: per tensor with a given scale (multiply by reciprocal) -- static, and pass 2 of dynamic per tensor
// MODE 2: absmax only: atomic max of rowmax/448 into *scale (pass 1 of dynamic per tensor)
// PARTS (MODE 0, rows of vectors): workgroups of a row, each with the maximum of all of it and the codes of the vectors i % PARTS = blockIdx.y of every thread.
template <typename T, int MODE, int TPB, int QV, int PARTS = 1>
__global__ __launch_bounds__(TPB) void fp8_quant_kernel(const T* __restrict__ in, int64_t in_stride,
                                                        uint8_t* __restrict__ out, int64_t out_stride,
                                                        float* __restrict__ scales, const float* __restrict__ scale_ub,
                                                        int hidden) {
  __shared__ float smem[TPB / 64];
  const int64_t row = blockIdx.x;
  const T* x = in + row * in_stride;
  uint8_t* y = out + row * out_stride;
  const int tid = threadIdx.x;

  const bool vec_ok = (hidden % 8 == 0) && (((uintptr_t)x % 16) == 0) && (((uintptr_t)y % 8) == 0) &&
                      (hidden <= TPB * QV * 8);
  Vec8<T> cache[QV];
  const float given = MODE == 1 ? *scales : 0.f;
  const int nvec = hidden / 8;

  if (vec_ok) {
#pragma unroll
    for (int i = 0; i < QV; ++i) {
      const int v = tid + i * TPB;
      if (v < nvec) cache[i].load(x + (int64_t)v * 8);
    }
  }

  float scale_or_inv;
  if constexpr (MODE != 1) {
    float amax = 0.f;
    if (vec_ok) {
#pragma unroll
      for (int i = 0; i < QV; ++i) {
        if (tid + i * TPB < nvec) {
          cache[i].unpack();
#pragma unroll
          for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(cache[i].f[e]));
        }
      }
    } else {
      for (int e = tid; e < hidden; e += TPB) amax = fmaxf(amax, fabsf(load_as_float<T>(x + e)));
    }
    amax = block_max<TPB>(amax, smem);
    if constexpr (MODE == 2) {
      // non-negative floats order like their bit patterns
      if (tid == 0) atomicMax(reinterpret_cast<int*>(scales), __float_as_int(amax / FP8_MAX));
      return;
    } else {
      float s = scale_ub ? fminf(amax, *scale_ub) : amax;
      s = fmaxf(s / FP8_MAX, 1.0f / (FP8_MAX * 512.0f));
      if (tid == 0 && (PARTS == 1 || blockIdx.y == 0)) scales[row] = s;
      scale_or_inv = s;
    }
  } else {
    scale_or_inv = 1.0f / given;
  }

  // MODE 0 on 16-bit inputs whose quotients cannot leave the normal range (no upper bound that could shrink the scale
  // below amax / 448, finite scale): the exact three-instruction division; the same for every thread of the row
  bool fast = false;
  float rcp = 0.f;
  if constexpr (MODE == 0 && sizeof(T) == 2) {
    fast = scale_ub == nullptr && scale_or_inv < __builtin_inff();
    rcp = 1.0f / scale_or_inv;
  }
  auto conv = [&](float v) -> float {
    if constexpr (MODE == 0) return clamp448(v / scale_or_inv);
    else return clamp448(v * scale_or_inv);
  };
  auto conv_fast = [&](float v) -> float { return clamp448(div16_exact(v, scale_or_inv, rcp)); };
  auto pack8 = [&](const float (&f)[8], auto&& cv) {
    v2u o;
    o.x = cvt2(cv(f[0]), cv(f[1])) | (cvt2(cv(f[2]), cv(f[3])) << 16);
    o.y = cvt2(cv(f[4]), cv(f[5])) | (cvt2(cv(f[6]), cv(f[7])) << 16);
    return o;
  };

  if (vec_ok) {
    if (fast) {
#pragma unroll
      for (int i = 0; i < QV; ++i) {
        const int v = tid + i * TPB;
        if (v < nvec && (PARTS == 1 || i % PARTS == (int)blockIdx.y)) *reinterpret_cast<v2u*>(y + (int64_t)v * 8) = pack8(cache[i].f, conv_fast);
      }
    } else {
#pragma unroll
      for (int i = 0; i < QV; ++i) {
        const int v = tid + i * TPB;
        if (v < nvec && (PARTS == 1 || i % PARTS == (int)blockIdx.y)) {
          if constexpr (MODE == 1) cache[i].unpack();
          *reinterpret_cast<v2u*>(y + (int64_t)v * 8) = pack8(cache[i].f, conv);
        }
      }
    }
  } else {
    for (int e = tid; e < hidden; e += TPB) y[e] = cvt1(conv(load_as_float<T>(x + e)));
  }
}

// Dynamic per token, one row per WAVEFRONT: the row (at most 64 lanes x NV vectors x 8 elements) sits in the wavefront's
// registers, the absmax is a butterfly over the lanes -- no LDS, no barrier, four rows per workgroup in flight
// independently.  Same arithmetic as MODE 0 above (the maximum is order-independent, the division is the IEEE one).
template <typename T, int NV>
__global__ __launch_bounds__(QTW) void fp8_quant_row_per_wave_kernel(const T* __restrict__ in, int64_t in_stride, int hidden, int rows,
                                                                     uint8_t* __restrict__ out, int64_t out_stride,
                                                                     float* __restrict__ scales, const float* __restrict__ scale_ub) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * (QTW / 64) + (threadIdx.x >> 6);
  if (row >= rows) return;
  const T* x = in + row * in_stride;
  uint8_t* y = out + row * out_stride;
  const int nvec = hidden / 8;
  Vec8<T> cache[NV];
  float amax = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int v = lane + i * 64;
    if (v < nvec) cache[i].load(x + (int64_t)v * 8);
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int v = lane + i * 64;
    if (v < nvec) {
      cache[i].unpack();
#pragma unroll
      for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(cache[i].f[e]));
    }
  }
  amax = wave_max(amax);
  float s = scale_ub ? fminf(amax, *scale_ub) : amax;
  s = fmaxf(s / FP8_MAX, 1.0f / (FP8_MAX * 512.0f));
  if (lane == 0) scales[row] = s;
  const bool fast = scale_ub == nullptr && s < __builtin_inff();      // see fp8_quant_kernel
  const float rcp = 1.0f / s;
  auto store8 = [&](int i, auto&& cv) {
    const int v = lane + i * 64;
    if (v < nvec) {
      float q[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) q[e] = clamp448(cv(cache[i].f[e]));
      v2u o;
      o.x = cvt2(q[0], q[1]) | (cvt2(q[2], q[3]) << 16);
      o.y = cvt2(q[4], q[5]) | (cvt2(q[6], q[7]) << 16);
      *reinterpret_cast<v2u*>(y + (int64_t)v * 8) = o;
    }
  };
  if (fast) {
#pragma unroll
    for (int i = 0; i < NV; ++i) store8(i, [&](float v) { return div16_exact(v, s, rcp); });
  } else {
#pragma unroll
    for (int i = 0; i < NV; ++i) store8(i, [&](float v) { return v / s; });
  }
}

// A given scale and rows without gaps: one run of elements, a vector of 8 to a thread, the last few elements one to a thread of the
// first workgroup.  Few rows are the latency of a load, which workgroups of one row each drew out by running on few compute units;
// short rows left most of a workgroup idle, and rows of a length that is no multiple of 8 went by single elements.
// Launch to launch, a workgroup per row -> this, us: 1 x 14336 2.35 -> 1.88, 16 x 14336 2.95 -> 1.85, 250 x 5120 2.88 -> 2.41, 333 x 3001
// 3.82 -> 2.24, 2048 x 4096 level, 4096 x 14336 32.3 -> 29.2, 8192 x 1024 7.3 -> 6.4, 30000 x 128 13.8 -> 3.9.
template <typename T>
__global__ __launch_bounds__(QT) void fp8_quant_run_kernel(const T* __restrict__ in, uint8_t* __restrict__ out,
                                                           const float* __restrict__ scale, int64_t total) {
  const float given = *scale;
  const int64_t nvec = total / 8, step = (int64_t)gridDim.x * blockDim.x;
  const int64_t first = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  Vec8<T> v;
  if (first < nvec) v.load(in + first * 8);
  const float inv = 1.0f / given;
  for (int64_t i = first; i < nvec; i += step) {
    if (i != first) v.load(in + i * 8);
    v.unpack();
    float q[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) q[e] = clamp448(v.f[e] * inv);
    v2u o;
    o.x = cvt2(q[0], q[1]) | (cvt2(q[2], q[3]) << 16);
    o.y = cvt2(q[4], q[5]) | (cvt2(q[6], q[7]) << 16);
    *reinterpret_cast<v2u*>(out + i * 8) = o;
  }
  const int64_t e = nvec * 8 + first;
  if (e < total) out[e] = cvt1(clamp448(load_as_float<T>(in + e) * inv));
}

// The first pass of the dynamic one over such a run: one atomic per workgroup instead of one per row -- they all meet at one address,
// about 12 ns each.  The whole dynamic call, us: 250 x 5120 9.1 -> 6.9, 1024 x 5120 20.4 -> 11.8, 4096 x 4096 60.7 -> 20.1, 8192 x
// 1024 103 -> 14.2, 4096 x 14336 86.5 -> 51.8; four workgroups of 256 to a compute unit 250 x 5120 12.6, 4096 x 4096 27.2.
template <typename T>
__global__ __launch_bounds__(QTA) void fp8_absmax_run_kernel(const T* __restrict__ in, float* __restrict__ scale, int64_t total) {
  __shared__ float smem[QTA / 64];
  const int64_t nvec = total / 8, step = (int64_t)gridDim.x * QTA;
  const int64_t first = (int64_t)blockIdx.x * QTA + threadIdx.x;
  float amax = 0.f;
  constexpr int AHEAD = 4;
  for (int64_t i = first; i < nvec; i += AHEAD * step) {
    Vec8<T> v[AHEAD];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
      if (i + u * step < nvec) v[u].load(in + (i + u * step) * 8);
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
      if (i + u * step < nvec) {
        v[u].unpack();
#pragma unroll
        for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(v[u].f[e]));
      }
  }
  const int64_t e = nvec * 8 + first;
  if (e < total) amax = fmaxf(amax, fabsf(load_as_float<T>(in + e)));
  amax = block_max<QTA>(amax, smem);
  if (threadIdx.x == 0) atomicMax(reinterpret_cast<int*>(scale), __float_as_int(amax / FP8_MAX));
}

__global__ void fill_zero_kernel(float* p) { *p = 0.f; }

// The row-per-wavefront kernel takes 16-bit rows of at most 4096 elements whose addresses allow 16-byte loads and
// 8-byte stores on every row (the caller only sends rows of up to 2048 elements).
static bool row_per_wave_ok(const void* in, int in_dtype, int64_t in_stride, const uint8_t* out, int64_t out_stride,
                            int64_t hidden) {
  return (in_dtype == VAQ_BF16 || in_dtype == VAQ_F16) && hidden % 8 == 0 && hidden <= 64 * 8 * 8 &&
         ((uintptr_t)in % 16) == 0 && in_stride % 8 == 0 && ((uintptr_t)out % 8) == 0 && out_stride % 8 == 0;
}

template <typename T>
static void launch_row_per_wave(const void* in, int64_t in_stride, uint8_t* out, int64_t out_stride, float* scales,
                                const float* ub, int64_t rows, int64_t hidden, hipStream_t s) {
  const dim3 grid((unsigned)((rows + QTW / 64 - 1) / (QTW / 64))), block(QTW);
  if (hidden <= 64 * 8 * 2)
    hipLaunchKernelGGL((fp8_quant_row_per_wave_kernel<T, 2>), grid, block, 0, s, (const T*)in, in_stride, (int)hidden, (int)rows, out,
                       out_stride, scales, ub);
  else if (hidden <= 64 * 8 * 4)
    hipLaunchKernelGGL((fp8_quant_row_per_wave_kernel<T, 4>), grid, block, 0, s, (const T*)in, in_stride, (int)hidden, (int)rows, out,
                       out_stride, scales, ub);
  else
    hipLaunchKernelGGL((fp8_quant_row_per_wave_kernel<T, 8>), grid, block, 0, s, (const T*)in, in_stride, (int)hidden, (int)rows, out,
                       out_stride, scales, ub);
}

template <int MODE, int TPB, int QV, int PARTS = 1>
static int launch_quant_tpb(const void* in, int in_dtype, int64_t in_stride, uint8_t* out, int64_t out_stride,
                            float* scales, const float* ub, int64_t rows, int64_t hidden, hipStream_t s) {
  const dim3 grid((unsigned)rows, PARTS), block(TPB);
  switch (in_dtype) {
    case VAQ_BF16:
      hipLaunchKernelGGL((fp8_quant_kernel<bf16_t, MODE, TPB, QV, PARTS>), grid, block, 0, s, (const bf16_t*)in, in_stride, out,
                         out_stride, scales, ub, (int)hidden);
      break;
    case VAQ_F16:
      hipLaunchKernelGGL((fp8_quant_kernel<f16_t, MODE, TPB, QV, PARTS>), grid, block, 0, s, (const f16_t*)in, in_stride, out,
                         out_stride, scales, ub, (int)hidden);
      break;
    case VAQ_F32:
      hipLaunchKernelGGL((fp8_quant_kernel<float, MODE, TPB, QV, PARTS>), grid, block, 0, s, (const float*)in, in_stride, out,
                         out_stride, scales, ub, (int)hidden);
      break;
    default:
      set_error("fp8_quant: unsupported input dtype tag %d", in_dtype);
      return VAQ_ERR_INVALID_ARG;
  }
  return VAQ_OK;
}

// Threads to a row and vectors of 8 elements to a thread.  One vector where 256 or 512 threads hold the row: the code is a third of
// that for four, and a launch of few rows is mostly latency (768 rows of 1024 / 2048 / 4096 per token: 3.3 / 3.5 / 3.9 -> 2.6 / 2.9 /
// 3.5 us, 16 rows of 4096 2.7 -> 2.4).  Many rows of up to 5120 elements run on 256 threads: twice the workgroups per compute unit,
// each a dependent chain of load, reduction and store of its own, and half the wavefronts in every barrier (4096 rows of 4096 / 5120:
// 10.7 / 12.6 us, 512 threads 12.4 / 14.2; 8192 wide 512 threads are ahead, 18.6 against 19.3).  Rows above 16384 take eight vectors
// to a thread instead of reading memory twice by single elements (one row of 20480 13.2 -> 3.4 us, 4096 of them 121 -> 39).
template <int MODE>
static int launch_quant(const void* in, int in_dtype, int64_t in_stride, uint8_t* out, int64_t out_stride,
                        float* scales, const float* ub, int64_t rows, int64_t hidden, hipStream_t s) {
  auto launch = [&](auto tpb, auto qv) {
    return launch_quant_tpb<MODE, decltype(tpb)::value, decltype(qv)::value>(in, in_dtype, in_stride, out, out_stride, scales, ub,
                                                                             rows, hidden, s);
  };
  const std::integral_constant<int, QT / 2> half;
  const std::integral_constant<int, QT> full;
  const std::integral_constant<int, 1> one;
  const std::integral_constant<int, 4> four;
  const std::integral_constant<int, 8> eight;
  // Rows that go by single elements are better off with many threads and few registers each: 512 rows or fewer of 1000 elements 20 %
  // ahead of 256 threads (256 x 1061 3.3 against 4.0 us), 802 rows of 32454 60 us with four vectors' registers, 88 with eight.
  const int64_t align = in_dtype == VAQ_F32 ? 4 : 8;      // elements of 16 bytes
  const bool strides_ok = rows == 1 || (in_stride % align == 0 && out_stride % 8 == 0);
  if (hidden % 8 != 0 || hidden > QT * 8 * 8 || (uintptr_t)in % 16 != 0 || (uintptr_t)out % 8 != 0 || !strides_ok)
    return rows >= 1024 && hidden <= 5120 ? launch(half, four) : launch(full, four);
  if (hidden <= QT / 2 * 8) return launch(half, one);
  if (rows >= 1024 && hidden <= 5120) return launch(half, four);
  if (hidden <= QT * 8) return launch(full, one);
  if constexpr (MODE == 0) {
    // Few long rows: four workgroups to a row, each with the row's maximum and the codes of one in four of a thread's vectors, the longer part of the arithmetic (rows of 8192
    // have two vectors to a thread, so that two of the workgroups find no codes; above 12288 each has some).  With the GEMM behind
    // it, us: 16 x 8192 10.20 -> 9.97, 16 / 64 x 14336 14.83 / 22.16 -> 14.50 / 21.81, 16 x 16384 18.34 -> 17.79; up to 6144 elements level.  Up to 8 rows a launch by itself takes
    // 0.1 us more and none less.  (Not where the codes go over the rows: another workgroup may still read them.)
    const uint64_t width = in_dtype == VAQ_F32 ? 4 : 2, last = (uint64_t)(rows - 1);
    const uint64_t i0 = (uintptr_t)in, i1 = i0 + (last * in_stride + hidden) * width, o0 = (uintptr_t)out, o1 = o0 + last * out_stride + hidden;
    if (hidden >= 8192 && hidden <= QT * 4 * 8 && rows > 8 && rows * 4 <= num_cus_current_device() && (o0 >= i1 || i0 >= o1))
      return launch_quant_tpb<MODE, QT, 4, 4>(in, in_dtype, in_stride, out, out_stride, scales, ub, rows, hidden, s);
  }
  return hidden <= QT * 4 * 8 ? launch(full, four) : launch(full, eight);
}

// MODE 1 (a given scale, also the second pass of the dynamic one) and 2 (its first): a run where the rows have no gaps.
template <int MODE>
static int launch_quant_per_tensor(const void* in, int in_dtype, int64_t in_stride, uint8_t* out, int64_t out_stride, float* scale,
                                   int64_t rows, int64_t hidden, hipStream_t s) {
  const bool run = (rows == 1 || (in_stride == hidden && (MODE == 2 || out_stride == hidden))) && (uintptr_t)in % 16 == 0 &&
                   (MODE == 2 || (uintptr_t)out % 8 == 0);
  if (!run) return launch_quant<MODE>(in, in_dtype, in_stride, out, out_stride, scale, nullptr, rows, hidden, s);
  // A given scale: up to eight workgroups of 256 to a compute unit, 512 threads beyond (16 x 14336 1.85 against 1.94 us; 2048 x 4096
  // 6.36 against 6.45); one vector to a thread, two are slower for few rows (250 x 5120 2.4 -> 2.6 us) and for many (4096 x 20480
  // 40 -> 42).  A launch of up to three workgroups takes 0.12 us less than one of four: 512 threads where that makes three of them
  // (2 x 4096 1.88 -> 1.74 us).  Maximum: at most one workgroup to a compute unit, two vectors to a thread where they are few.
  const int64_t total = rows * hidden, vecs = total / 8, cus = num_cus_current_device();
  const bool three = vecs > 3 * (QT / 2) && vecs <= 3 * QT;
  const int threads = MODE == 2 ? QTA : vecs <= cus * 2048 && !three ? QT / 2 : QT;
  const int64_t share = MODE == 2 ? 2 * QTA : threads, cap = MODE == 2 ? cus : cus * 32 * QT / threads;
  const int64_t blocks = (vecs + share - 1) / share;
  const dim3 grid((unsigned)(blocks < 1 ? 1 : blocks < cap ? blocks : cap)), block(threads);
  auto launch = [&](auto tag) {
    using T = decltype(tag);
    if constexpr (MODE == 1) hipLaunchKernelGGL(fp8_quant_run_kernel<T>, grid, block, 0, s, (const T*)in, out, scale, total);
    else hipLaunchKernelGGL(fp8_absmax_run_kernel<T>, grid, block, 0, s, (const T*)in, scale, total);
    return VAQ_OK;
  };
  if (in_dtype == VAQ_BF16) return launch(bf16_t{});
  if (in_dtype == VAQ_F16) return launch(f16_t{});
  if (in_dtype == VAQ_F32) return launch(float{});
  set_error("fp8_quant: unsupported input dtype tag %d", in_dtype);
  return VAQ_ERR_INVALID_ARG;
}

static int check_quant(const char* who, const void* in, int64_t in_stride, const uint8_t* out, int64_t out_stride,
                       const float* scale, int64_t rows, int64_t hidden) {
  VAQ_CHECK_ARG(rows >= 0 && hidden > 0, "%s: bad shape [%lld, %lld]", who, (long long)rows, (long long)hidden);
  VAQ_CHECK_ARG(rows < (1ll << 31) && hidden < (1ll << 31), "%s: shape too large", who);
  VAQ_CHECK_ARG(in_stride >= hidden && out_stride >= hidden, "%s: row strides (%lld, %lld) smaller than hidden = %lld",
                who, (long long)in_stride, (long long)out_stride, (long long)hidden);
  if (rows > 0) VAQ_CHECK_ARG(in && out && scale, "%s: null pointer", who);
  return VAQ_OK;
}

}  // namespace vaq

extern "C" int vaq_fp8_quant_per_token(const void* in, int in_dtype, int64_t in_row_stride, uint8_t* out,
                                       int64_t out_row_stride, float* scales, const float* scale_ub, int64_t rows,
                                       int64_t hidden, void* stream) {
  return vaq_fp8_quant_per_token_tuned(in, in_dtype, in_row_stride, out, out_row_stride, scales, scale_ub, rows, hidden,
                                       stream, nullptr);
}

extern "C" int vaq_fp8_quant_per_token_tuned(const void* in, int in_dtype, int64_t in_row_stride, uint8_t* out,
                                             int64_t out_row_stride, float* scales, const float* scale_ub, int64_t rows,
                                             int64_t hidden, void* stream, const VaqTuning* tuning_or_null) {
  using namespace vaq;
  const TuningScope scope(tuning_or_null);
  int rc = check_quant("fp8_quant_per_token", in, in_row_stride, out, out_row_stride, scales, rows, hidden);
  if (rc != VAQ_OK || rows == 0) return rc;
  // Measured: a row per wavefront is 1.1-1.6x faster for short rows in large batches; with few rows a whole workgroup
  // per row has the shorter latency, and from 4096 elements on the 64 registers of row data per lane cost more than the
  // barriers saved.
  const bool many_short_rows = hidden <= 1024 ? rows >= 1024 : (hidden <= 2048 && rows >= 2048);
  const int force = tuning().quant_wg_per_row;      // 1: a workgroup per row, 2: a wavefront per row where it can run
  if ((force == 2 || (force == 0 && many_short_rows)) &&
      row_per_wave_ok(in, in_dtype, in_row_stride, out, out_row_stride, hidden)) {
    if (in_dtype == VAQ_BF16)
      launch_row_per_wave<bf16_t>(in, in_row_stride, out, out_row_stride, scales, scale_ub, rows, hidden, (hipStream_t)stream);
    else
      launch_row_per_wave<f16_t>(in, in_row_stride, out, out_row_stride, scales, scale_ub, rows, hidden, (hipStream_t)stream);
  } else {
    rc = launch_quant<0>(in, in_dtype, in_row_stride, out, out_row_stride, scales, scale_ub, rows, hidden,
                         (hipStream_t)stream);
    if (rc != VAQ_OK) return rc;
  }
  VAQ_CHECK_LAUNCH("fp8_quant_per_token");
  return VAQ_OK;
}

extern "C" int vaq_fp8_quant_static(const void* in, int in_dtype, int64_t in_row_stride, uint8_t* out,
                                    int64_t out_row_stride, const float* scale, int64_t rows, int64_t hidden,
                                    void* stream) {
  using namespace vaq;
  int rc = check_quant("fp8_quant_static", in, in_row_stride, out, out_row_stride, scale, rows, hidden);
  if (rc != VAQ_OK || rows == 0) return rc;
  rc = launch_quant_per_tensor<1>(in, in_dtype, in_row_stride, out, out_row_stride, const_cast<float*>(scale), rows, hidden,
                                  (hipStream_t)stream);
  if (rc != VAQ_OK) return rc;
  VAQ_CHECK_LAUNCH("fp8_quant_static");
  return VAQ_OK;
}

extern "C" int vaq_fp8_quant_dynamic(const void* in, int in_dtype, int64_t in_row_stride, uint8_t* out,
                                     int64_t out_row_stride, float* scale, int64_t rows, int64_t hidden,
                                     void* stream) {
  using namespace vaq;
  int rc = check_quant("fp8_quant_dynamic", in, in_row_stride, out, out_row_stride, scale, rows, hidden);
  if (rc != VAQ_OK || rows == 0) return rc;
  hipStream_t s = (hipStream_t)stream;
  // the running maximum starts from zero; a one-thread kernel rather than a memset node keeps the call graph-capturable
  hipLaunchKernelGGL(fill_zero_kernel, dim3(1), dim3(1), 0, s, scale);
  rc = launch_quant_per_tensor<2>(in, in_dtype, in_row_stride, out, out_row_stride, scale, rows, hidden, s);
  if (rc != VAQ_OK) return rc;
  rc = launch_quant_per_tensor<1>(in, in_dtype, in_row_stride, out, out_row_stride, scale, rows, hidden, s);
  if (rc != VAQ_OK) return rc;
  VAQ_CHECK_LAUNCH("fp8_quant_dynamic");
  return VAQ_OK;
}
