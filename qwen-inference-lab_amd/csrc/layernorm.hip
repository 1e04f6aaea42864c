// Norms fused with a scaled residual add: layer norm (mean removed, weight, optional bias) and RMS norm.
// The residual stream is float32; statistics, the sum and the weight product are float32, the result is rounded once.
#include "common.h"
#include "operand.h"
#include "partials.h"

template <typename TD>
__device__ __forceinline__ float row_value(const float* __restrict__ x, const TD* __restrict__ delta, size_t at, int i,
                                           int splits, size_t stride, float delta_scale) {
  float v = x[i];
  if (delta) v = v + delta_scale * parts_sum(delta, at + i, splits, stride);
  return v;
}

// One block per output row m; r = rows ? rows[m] : m.
//   v = stream[r] + delta_scale * delta[r];  if (update) stream[r] = v;
//   CENTRE: out[m] = (v - mean(v)) / sqrt(mean((v - mean(v))^2) + eps) * weight (+ bias)
//   else:   out[m] = v / sqrt(mean(v^2) + eps) * weight (+ bias)
template <typename TD, typename T, int CENTRE>
__global__ void add_norm_kernel(float* __restrict__ stream, const TD* __restrict__ delta, int splits, size_t split_stride,
                                float delta_scale, const int* __restrict__ rows, const float* __restrict__ weight,
                                const float* __restrict__ bias, T* __restrict__ out, int width, float eps, int update) {
  __shared__ float scratch[16];
  const int m = blockIdx.x;
  const size_t r = rows ? (size_t)rows[m] : (size_t)m;
  float* x = stream + r * width;
  const size_t at = r * width;
  float sum = 0.f;
  for (int i = threadIdx.x; i < width; i += blockDim.x) {
    const float v = row_value(x, delta, at, i, splits, split_stride, delta_scale);
    if (delta && update) x[i] = v;
    sum += v;
  }
  const TD* later = update ? nullptr : delta;          // after the update the stream holds the sum already
  float mean = 0.f;
  if (CENTRE) mean = block_sum(sum, scratch) / (float)width;
  float squares = 0.f;
  for (int i = threadIdx.x; i < width; i += blockDim.x) {
    const float c = row_value(x, later, at, i, splits, split_stride, delta_scale) - mean;
    squares += c * c;
  }
  squares = block_sum(squares, scratch);
  const float scale = 1.f / sqrtf(squares / (float)width + eps);
  T* y = out + (size_t)m * width;
  for (int i = threadIdx.x; i < width; i += blockDim.x) {
    const float c = row_value(x, later, at, i, splits, split_stride, delta_scale) - mean;
    st(y + i, c * scale * weight[i] + (bias ? bias[i] : 0.f));
  }
}

// The same with the row in registers (width % 4 == 0, at most 4 * J * THREADS, 16-byte aligned operands): 16-byte accesses
// and one pass over memory where the kernel above makes three of 4 bytes a lane; what is added waits for its own loads, partial
// sums four at a time (operand_at4).  Bound by memory with many rows and by the waits for it with few (3,044 rows of 2,048 in bfloat16
// 27 -> 17 us, 8 rows with four partial sums 9.5 -> 4.1).
template <typename TD, typename T, int CENTRE, int THREADS, int J>
__global__ void __launch_bounds__(THREADS)
add_norm_vec_kernel(float* __restrict__ stream, const TD* __restrict__ delta, int splits, size_t split_stride, float delta_scale,
                    const int* __restrict__ rows, const float* __restrict__ weight, const float* __restrict__ bias,
                    T* __restrict__ out, int width, float eps, int update) {
  __shared__ float scratch[16];
  const int m = blockIdx.x;
  const size_t r = rows ? (size_t)rows[m] : (size_t)m;
  float* x = stream + r * width;
  const Operand operand{delta, sizeof(TD) == 2 ? QIL_BF16 : QIL_F32, splits, split_stride};
  const float4 none = make_float4(0.f, 0.f, 0.f, 0.f);
  float4 v[J], w[J], b[J];
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int i = (threadIdx.x + j * THREADS) * 4;
    const bool live = i < width;
    v[j] = live ? ld4(x + i) : none;
    w[j] = live ? ld4(weight + i) : none;
    b[j] = live && bias ? ld4(bias + i) : none;
    if (live && delta) {
      const float4 d = operand_at4(operand, r * width + i);
      v[j] = make_float4(v[j].x + delta_scale * d.x, v[j].y + delta_scale * d.y, v[j].z + delta_scale * d.z, v[j].w + delta_scale * d.w);
      if (update) st4(x + i, v[j]);
    }
    sum += (v[j].x + v[j].y) + (v[j].z + v[j].w);
  }
  const float mean = CENTRE ? block_sum(sum, scratch) / (float)width : 0.f;
  float squares = 0.f;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    if ((threadIdx.x + j * THREADS) * 4 < width) {
      v[j] = make_float4(v[j].x - mean, v[j].y - mean, v[j].z - mean, v[j].w - mean);
      squares += (v[j].x * v[j].x + v[j].y * v[j].y) + (v[j].z * v[j].z + v[j].w * v[j].w);
    }
  }
  squares = block_sum(squares, scratch);
  const float scale = 1.f / sqrtf(squares / (float)width + eps);
  T* y = out + (size_t)m * width;
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int i = (threadIdx.x + j * THREADS) * 4;
    if (i < width)
      st4(y + i, make_float4(v[j].x * scale * w[j].x + b[j].x, v[j].y * scale * w[j].y + b[j].y, v[j].z * scale * w[j].z + b[j].z,
                             v[j].w * scale * w[j].w + b[j].w));
  }
}

extern "C" {

// delta: null, or the sub-layer output to add: delta_dtype QIL_BF16 (one array, splits == 1) or QIL_F32
// ([splits][delta_rows][width] partial sums).  centre: 1 layer norm, 0 RMS norm.  bias: float32 [width] or null.
// out_dtype: type of `out`.
int qil_add_norm(float* stream, const void* delta, int delta_dtype, int splits, int delta_rows, float delta_scale,
                 const int* rows, const float* weight, const float* bias, void* out, int n_out, int width, float eps, int update, int centre,
                 int out_dtype, hipStream_t s) {
  if (n_out == 0) return 0;
  if (width < 1 || splits < 1 || (delta_dtype == QIL_BF16 && splits != 1)) return -1;
  const size_t stride = (size_t)delta_rows * width;
  const int threads = width >= 2048 ? 512 : width >= 512 ? 256 : width >= 128 ? 128 : 64;
  const bool vec = width % 4 == 0 && width <= 8192 &&
                   (((uintptr_t)stream | (uintptr_t)delta | (uintptr_t)weight | (uintptr_t)bias | (uintptr_t)out) % 16 == 0);
#define QIL_NORM_VEC(TD, T, C, THREADS, J)                                                                            \
  hipLaunchKernelGGL((add_norm_vec_kernel<TD, T, C, THREADS, J>), dim3(n_out), dim3(THREADS), 0, s, stream,            \
                     (const TD*)delta, splits, stride, delta_scale, rows, weight, bias, (T*)out, width, eps, update)
#define QIL_NORM_LAUNCH(TD, T, C)                                                                                     \
  do {                                                                                                                \
    if (vec && width <= 256) QIL_NORM_VEC(TD, T, C, 64, 1);                                                           \
    else if (vec && width <= 1024) QIL_NORM_VEC(TD, T, C, 256, 1);                                                    \
    else if (vec && width <= 2048) QIL_NORM_VEC(TD, T, C, 512, 1);                                                    \
    else if (vec && width <= 4096) QIL_NORM_VEC(TD, T, C, 512, 2);                                                    \
    else if (vec) QIL_NORM_VEC(TD, T, C, 1024, 2);                                                                    \
    else                                                                                                              \
      hipLaunchKernelGGL((add_norm_kernel<TD, T, C>), dim3(n_out), dim3(threads), 0, s, stream, (const TD*)delta,     \
                         splits, stride, delta_scale, rows, weight, bias, (T*)out, width, eps, update);               \
  } while (0)
#define QIL_NORM_CASE(TD, T) do { if (centre) QIL_NORM_LAUNCH(TD, T, 1); else QIL_NORM_LAUNCH(TD, T, 0); } while (0)
  if (out_dtype == QIL_F32) {
    if (delta_dtype != QIL_F32) return -1;
    QIL_NORM_CASE(float, float);
  } else if (delta_dtype == QIL_F32) {
    QIL_NORM_CASE(float, bf16_t);
  } else {
    QIL_NORM_CASE(bf16_t, bf16_t);
  }
#undef QIL_NORM_CASE
#undef QIL_NORM_LAUNCH
#undef QIL_NORM_VEC
  QIL_RETURN_LAUNCH_STATUS();
}

}  // extern "C"
