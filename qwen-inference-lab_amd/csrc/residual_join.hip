// What the sub-layers of a layer with gated branches leave joins the float32 residual stream, fused with the RMS norm
// that follows:
//     x = stream[r] + sigmoid(g1 + b1) * (a_scale * a + b_scale * b) + sigmoid(g2 + b2) * f + plus[r] + step
//     if (update) stream[r] = x
//     out[m] = x / sqrt(mean(x^2) + eps) * weight
// with r = rows ? rows[m] : m.  a, b: the mixer's output, or the outputs of two mixers side by side (b optional); f: the
// feed-forward's output (optional).  g1, g2: the gates' logits (columns [0, width) and [width, 2 width) of the operand
// `gates`) with stored biases b1, b2 behind one another; without gates the factors are 1.  plus float32 [.., width] and
// step float32 [width]: what a pass of a loop over layers adds before its first layer (optional).  Every operand is an
// array of the model's type or float32 partial sums (operand.h).  Everything is float32 until the one rounding of `out`.
// One block a row; the row waits in LDS between the sum and the norm.
#include "common.h"
#include "operand.h"

struct JoinInputs {
  Operand a, b, f, gates;                                  // data null: not there
  size_t a_row, b_row, f_row, g_row;                       // elements between two rows
  float a_scale, b_scale;
  const float* bias;                                       // [2 width] (or [width] without f)
  const float* plus;
  const float* step;
};

template <int V> __device__ __forceinline__ void join_load(const Operand& x, size_t at, float* v) {
  if constexpr (V == 4) {
    const float4 q = operand_at4(x, at);
    v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
  } else {
    v[0] = operand_at(x, at);
  }
}
template <int V> __device__ __forceinline__ void join_floats(const float* p, float* v) {
  if constexpr (V == 4) {
    const float4 q = ld4(p);
    v[0] = q.x; v[1] = q.y; v[2] = q.z; v[3] = q.w;
  } else {
    v[0] = p[0];
  }
}

template <typename T, int V>
__global__ void residual_join_kernel(float* __restrict__ stream, JoinInputs in, const int* __restrict__ rows,
                                     const float* __restrict__ weight, T* __restrict__ out, int width, float eps, int update) {
  extern __shared__ __align__(16) float held[];            // [width]
  __shared__ float scratch[16];
  const int m = blockIdx.x;
  const size_t r = rows ? (size_t)rows[m] : (size_t)m;
  float* x = stream + r * width;
  float squares = 0.f;
  for (int i = threadIdx.x * V; i < width; i += blockDim.x * V) {
    float v[V], t[V], u[V];
    join_floats<V>(x + i, v);
    if (in.a.data) {
      join_load<V>(in.a, r * in.a_row + i, t);
#pragma unroll
      for (int e = 0; e < V; ++e) t[e] *= in.a_scale;
      if (in.b.data) {
        join_load<V>(in.b, r * in.b_row + i, u);
#pragma unroll
        for (int e = 0; e < V; ++e) t[e] += in.b_scale * u[e];
      }
      if (in.gates.data) {
        float b[V];
        join_load<V>(in.gates, r * in.g_row + i, u);
        join_floats<V>(in.bias + i, b);
#pragma unroll
        for (int e = 0; e < V; ++e) t[e] = t[e] / (1.f + expf(-(u[e] + b[e])));
      }
      if (in.f.data) {
        float f[V];
        join_load<V>(in.f, r * in.f_row + i, f);
        if (in.gates.data) {
          float b[V];
          join_load<V>(in.gates, r * in.g_row + width + i, u);
          join_floats<V>(in.bias + width + i, b);
#pragma unroll
          for (int e = 0; e < V; ++e) f[e] = f[e] / (1.f + expf(-(u[e] + b[e])));
        }
#pragma unroll
        for (int e = 0; e < V; ++e) t[e] += f[e];
      }
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] += t[e];
    }
    if (in.plus) {
      join_floats<V>(in.plus + r * width + i, u);
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] += u[e];
    }
    if (in.step) {
      join_floats<V>(in.step + i, u);
#pragma unroll
      for (int e = 0; e < V; ++e) v[e] += u[e];
    }
#pragma unroll
    for (int e = 0; e < V; ++e) {
      held[i + e] = v[e];
      squares += v[e] * v[e];
    }
    if (update) {
      if constexpr (V == 4) st4(x + i, make_float4(v[0], v[1], v[2], v[3]));
      else x[i] = v[0];
    }
  }
  squares = block_sum(squares, scratch);
  const float unit = 1.f / sqrtf(squares / (float)width + eps);
  T* y = out + (size_t)m * width;
  for (int i = threadIdx.x * V; i < width; i += blockDim.x * V) {      // (a thread meets its own elements again)
    if constexpr (V == 4) {
      const float4 w = ld4(weight + i);
      st4(y + i, make_float4(held[i] * unit * w.x, held[i + 1] * unit * w.y, held[i + 2] * unit * w.z, held[i + 3] * unit * w.w));
    } else {
      st(y + i, held[i] * unit * weight[i]);
    }
  }
}

// Plain operands of bfloat16 (the products of many rows), all of them there but b: eight columns a thread, every operand asked
// for before one is taken, the row in registers.  Where each operand's kind is found out at run time its load waits inside its
// branch: 2,048 rows of 2,048 columns, two mixers and a feed-forward, 23.0 -> 19.4 us (84 MB; the quotients and exponentials of
// the gates are about 6 of them).  blockDim.x = width / 8.
template <bool TWO>
__global__ void __launch_bounds__(1024)
residual_join_plain_kernel(float* __restrict__ stream, const bf16_t* __restrict__ a, const bf16_t* __restrict__ b,
                           const bf16_t* __restrict__ f, const bf16_t* __restrict__ gates, int a_row, int b_row, int f_row,
                           int g_row, float a_scale, float b_scale, const float* __restrict__ bias,
                           const float* __restrict__ weight, bf16_t* __restrict__ out, int width, float eps) {
  __shared__ float scratch[16];
  const size_t m = blockIdx.x;
  const int i = threadIdx.x * 8;
  float* x = stream + m * width + i;
  float v[8], t[8], u[8], y[8], g1[8], g2[8], b1[8], b2[8], w[8];
  ld8(x, v);
  ld8(a + m * a_row + i, t);
  if (TWO) ld8(b + m * b_row + i, u);
  ld8(f + m * f_row + i, y);
  ld8(gates + m * g_row + i, g1);
  ld8(gates + m * g_row + width + i, g2);
  ld8(bias + i, b1);
  ld8(bias + width + i, b2);
  ld8(weight + i, w);
  float squares = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    float mixed = t[e] * a_scale;
    if (TWO) mixed += b_scale * u[e];
    mixed = mixed / (1.f + expf(-(g1[e] + b1[e])));
    mixed += y[e] / (1.f + expf(-(g2[e] + b2[e])));
    v[e] += mixed;
    squares += v[e] * v[e];
  }
  st4(x, make_float4(v[0], v[1], v[2], v[3]));
  st4(x + 4, make_float4(v[4], v[5], v[6], v[7]));
  squares = block_sum(squares, scratch);
  const float unit = 1.f / sqrtf(squares / (float)width + eps);
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = v[e] * unit * w[e];
  *reinterpret_cast<uint4*>(out + m * width + i) =
      make_uint4(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7]));
}

extern "C" {

// a, b, f, gates: (pointer or null, code, splits, elements of a row); the split stride is total_rows times the row.
// out [n_out, width] of out_dtype.
int qil_residual_join(float* stream, const void* a, int a_code, int a_splits, int a_row, float a_scale, const void* b,
                      int b_code, int b_splits, int b_row, float b_scale, const void* f, int f_code, int f_splits, int f_row,
                      const void* gates, int g_code, int g_splits, int g_row, const float* bias, const float* plus,
                      const float* step, const int* rows, const float* weight, void* out, int n_out, int total_rows,
                      int width, float eps, int update, int out_dtype, hipStream_t s) {
  if (n_out == 0) return 0;
  if (width < 1 || !weight || !out || (b && !a) || (f && !a) || (gates && !bias) || (gates && !a)) return -1;
  const void* data[4] = {a, b, f, gates};
  const int codes[4] = {a_code, b_code, f_code, g_code}, splits[4] = {a_splits, b_splits, f_splits, g_splits};
  const int row[4] = {a_row, b_row, f_row, g_row};
  JoinInputs in;
  Operand* ops[4] = {&in.a, &in.b, &in.f, &in.gates};
  bool vec = width % 4 == 0;
  for (int k = 0; k < 4; ++k) {
    if (data[k] && (splits[k] < 1 || (codes[k] == QIL_BF16 && splits[k] != 1) || row[k] < (k == 3 && f ? 2 * width : width)))
      return -1;
    *ops[k] = Operand{data[k], codes[k], splits[k], (size_t)total_rows * row[k]};
    vec = vec && (!data[k] || (row[k] % 4 == 0 && (uintptr_t)data[k] % 16 == 0));
  }
  in.a_row = a_row; in.b_row = b_row; in.f_row = f_row; in.g_row = g_row;
  in.a_scale = a_scale; in.b_scale = b_scale;
  in.bias = bias; in.plus = plus; in.step = step;
  vec = vec && (((uintptr_t)stream | (uintptr_t)bias | (uintptr_t)plus | (uintptr_t)step | (uintptr_t)weight | (uintptr_t)out) % 16) == 0;
  const size_t lds = (size_t)width * sizeof(float);
  if (lds > 128 * 1024) return -1;
  // whole waves of eight columns a thread, up to 1,024 threads; other widths, kinds and partial sums: the general kernel
  bool plain = vec && out_dtype == QIL_BF16 && a && f && gates && !plus && !step && !rows && update && width % 512 == 0 && width <= 8192;
  for (int k = 0; k < 4; ++k) plain = plain && (!data[k] || (codes[k] == QIL_BF16 && row[k] % 8 == 0));
  if (plain) {
#define QIL_JOIN_PLAIN(TWO)                                                                                           \
  hipLaunchKernelGGL(residual_join_plain_kernel<TWO>, dim3(n_out), dim3(width / 8), 0, s, stream, (const bf16_t*)a,    \
                     (const bf16_t*)b, (const bf16_t*)f, (const bf16_t*)gates, a_row, b_row, f_row, g_row, a_scale,    \
                     b_scale, bias, weight, (bf16_t*)out, width, eps)
    if (b) QIL_JOIN_PLAIN(true);
    else QIL_JOIN_PLAIN(false);
#undef QIL_JOIN_PLAIN
    QIL_RETURN_LAUNCH_STATUS();
  }
  const int lanes = vec ? width / 4 : width;
  const int threads = lanes >= 1024 ? 1024 : (lanes + 63) / 64 * 64;
#define QIL_JOIN(T, V)                                                                                               \
  do {                                                                                                               \
    if (lds > 60 * 1024) {                                                                                           \
      hipError_t e = hipFuncSetAttribute((const void*)residual_join_kernel<T, V>,                                    \
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);                      \
      if (e != hipSuccess) return (int)e;                                                                            \
    }                                                                                                                \
    hipLaunchKernelGGL((residual_join_kernel<T, V>), dim3(n_out), dim3(threads), lds, s, stream, in, rows, weight,    \
                       (T*)out, width, eps, update);                                                                 \
  } while (0)
  if (out_dtype == QIL_F32) { if (vec) QIL_JOIN(float, 4); else QIL_JOIN(float, 1); }
  else { if (vec) QIL_JOIN(bf16_t, 4); else QIL_JOIN(bf16_t, 1); }
#undef QIL_JOIN
  QIL_RETURN_LAUNCH_STATUS();
}

}  // extern "C"
