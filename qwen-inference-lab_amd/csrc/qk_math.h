// Eight consecutive elements of a head at a time: the sum of a product's partial results, the head's
// RMSNorm and the rotation by position, as the vector kernel of qk_rope.hip and the fused decode
// attention (attention_decode.hip) both do them.  One source for both, so that a query or key comes out
// bit for bit the same whichever kernel made it.
#pragma once
#include "common.h"

// What a query at `position` is multiplied by when its temperature grows with the logarithm of the position:
// 1 + coef * ln(floor((position + 1) / every) + 1); every <= 0: 1.
__device__ __forceinline__ float query_temperature(int position, float coef, int every) {
  return every > 0 ? 1.f + coef * logf((float)((position + 1) / every) + 1.f) : 1.f;
}

// The projection's bias (float32, by column of the product; null: none) joins eight summed elements.
__device__ __forceinline__ void add_bias8(float (&x)[8], const float* __restrict__ bias, int column) {
  if (!bias) return;
  const float4 lo = *reinterpret_cast<const float4*>(bias + column), hi = *reinterpret_cast<const float4*>(bias + column + 4);
  x[0] += lo.x; x[1] += lo.y; x[2] += lo.z; x[3] += lo.w; x[4] += hi.x; x[5] += hi.y; x[6] += hi.z; x[7] += hi.w;
}

__device__ __forceinline__ void load8_sum(const float* base, size_t index, int splits, size_t stride, float* out) {
#pragma unroll
  for (int e = 0; e < 8; ++e) out[e] = 0.f;
  for (int s0 = 0; s0 < splits; s0 += 4) {
    float4 lo[4], hi[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float* p = base + (size_t)min(s0 + u, splits - 1) * stride + index;
      lo[u] = *reinterpret_cast<const float4*>(p);
      hi[u] = *reinterpret_cast<const float4*>(p + 4);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
      if (s0 + u < splits) {
        out[0] += lo[u].x; out[1] += lo[u].y; out[2] += lo[u].z; out[3] += lo[u].w;
        out[4] += hi[u].x; out[5] += hi[u].y; out[6] += hi[u].z; out[7] += hi[u].w;
      }
  }
}
__device__ __forceinline__ void load8_sum(const bf16_t* base, size_t index, int, size_t, float* out) { ld8(base + index, out); }
// The same sum (the same order of additions) with the loads of eight splits in flight at a time: for a
// kernel in which this is a wave's only work before a barrier.
__device__ __forceinline__ void load8_sum_wide(const float* base, size_t index, int splits, size_t stride, float* out) {
#pragma unroll
  for (int e = 0; e < 8; ++e) out[e] = 0.f;
  for (int s0 = 0; s0 < splits; s0 += 8) {
    float4 lo[8], hi[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float* p = base + (size_t)min(s0 + u, splits - 1) * stride + index;
      lo[u] = *reinterpret_cast<const float4*>(p);
      hi[u] = *reinterpret_cast<const float4*>(p + 4);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (s0 + u < splits) {
        out[0] += lo[u].x; out[1] += lo[u].y; out[2] += lo[u].z; out[3] += lo[u].w;
        out[4] += hi[u].x; out[5] += hi[u].y; out[6] += hi[u].z; out[7] += hi[u].w;
      }
  }
}
__device__ __forceinline__ void store8(float* p, const float* v) {
  *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  *reinterpret_cast<float4*>(p + 4) = make_float4(v[4], v[5], v[6], v[7]);
}
__device__ __forceinline__ void store8(bf16_t* p, const float* v) {
  *reinterpret_cast<uint4*>(p) = make_uint4(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7]));
}

// A head of d elements is spread over TG = d / 8 lanes of a wave (a power of two; lane's chunk = its 8
// elements); every lane of the group must call.  x: the elements, replaced by the result (float32, to
// be rounded to T when stored).  weight: null = no norm.  cos_table: null = no rotation; rot: rotated
// width, pairs (i, i + rot / 2), rot / 16 a power of two.  d: the number of elements the norm's mean runs over.
// sin_table null with a cos_table: the latter holds the rot / 2 frequencies, and the angle position * frequency,
// its cosine and its sine are made here in float32 (no table bounds the positions).
// rotate_first: the rotation comes before the norm (a design that norms what it has rotated).
// (qil/model.py:15-23, 42-46, 52-55)
// What eight elements of a head are normed and turned with: the norm's weights, and the cosines and sines of their pairs
// (chunks in the rotated part).  Loading them is apart from using them, for a kernel that asks for all it needs first.
struct HeadFactors {
  float w[8], c[8], sn[8];
};
__device__ __forceinline__ void load_eight(const float* p, float (&to)[8]) {
  const float4 lo = *reinterpret_cast<const float4*>(p), hi = *reinterpret_cast<const float4*>(p + 4);
  to[0] = lo.x; to[1] = lo.y; to[2] = lo.z; to[3] = lo.w; to[4] = hi.x; to[5] = hi.y; to[6] = hi.z; to[7] = hi.w;
}
// FREQUENCIES: 1 made from frequencies, 0 read from tables, -1 as the arguments say (a kernel that knows does not carry the code
// for both: eight sines and cosines are 10 KB, and kernels of a few us wait for the instruction cache).
template <int FREQUENCIES = -1>
__device__ __forceinline__ void load_turns(HeadFactors& f, int chunk, const float* __restrict__ cos_table,
                                           const float* __restrict__ sin_table, int position, int rot) {
  const int half_chunks = rot >> 4;                   // chunks in half of the rotated width (a power of two)
  if (chunk < 2 * half_chunks) {
    const int pair = chunk < half_chunks ? chunk : chunk - half_chunks;
    if (FREQUENCIES == 0 || (FREQUENCIES < 0 && sin_table)) {
      const size_t at = (size_t)position * (rot >> 1) + pair * 8;
      load_eight(cos_table + at, f.c);
      load_eight(sin_table + at, f.sn);
    } else {
      const float* freq = cos_table + pair * 8;
#pragma unroll
      for (int e = 0; e < 8; ++e) sincosf((float)position * freq[e], &f.sn[e], &f.c[e]);
    }
  }
}
template <typename T>
__device__ __forceinline__ void head_norm8(float (&x)[8], int TG, const HeadFactors& f, int d, float eps) {
  float sum = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) sum += x[e] * x[e];
  if (TG == 16) {                                       // rows of the data-parallel moves: the same additions without trips through LDS
    sum += lane_move<0x128>(sum);                       // rotated by 8: the lane ^ 8
    sum += lane_move<0x124>(sum);                       // by 4 (eight lanes agree with the other eight by now)
    sum += lane_move<0x4E>(sum);
    sum += lane_move<0xB1>(sum);
  } else {
    for (int o = TG >> 1; o > 0; o >>= 1) sum += __shfl_xor(sum, o, QIL_WAVE);
  }
  const float rstd = rsqrtf(sum / (float)d + eps);
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = round_to<T>(x[e] * rstd) * f.w[e];
}
__device__ __forceinline__ void rotate8(float (&x)[8], int chunk, const HeadFactors& f, int rot) {
  const int half_chunks = rot >> 4;
  float other[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) other[e] = __shfl_xor(x[e], half_chunks, QIL_WAVE);
  if (chunk < 2 * half_chunks) {
    const bool first = chunk < half_chunks;
#pragma unroll
    for (int e = 0; e < 8; ++e)                         // (which product is rounded alone is written out: the same in every kernel)
      x[e] = fmaf(x[e], f.c[e], first ? -(other[e] * f.sn[e]) : other[e] * f.sn[e]);
  }
}
template <typename T>
__device__ __forceinline__ void norm_rope8(float (&x)[8], int chunk, int TG, const HeadFactors& f, bool norms, int d, float eps,
                                           bool rotates, int rot, bool rotate_first) {
  if (rotates && rotate_first) rotate8(x, chunk, f, rot);
  if (norms) head_norm8<T>(x, TG, f, d, eps);
  if (rotates && !rotate_first) rotate8(x, chunk, f, rot);
}
template <typename T>
__device__ __forceinline__ void norm_rope8(float (&x)[8], int chunk, int TG, const float* __restrict__ weight, int d,
                                           float eps, const float* __restrict__ cos_table,
                                           const float* __restrict__ sin_table, int position, int rot,
                                           bool rotate_first = false) {
  const bool rotates = cos_table && rot > 0;
  HeadFactors f;
  if (weight) load_eight(weight + chunk * 8, f.w);
  if (rotates) load_turns(f, chunk, cos_table, sin_table, position, rot);
  norm_rope8<T>(x, chunk, TG, f, weight != nullptr, d, eps, rotates, rot, rotate_first);
}
