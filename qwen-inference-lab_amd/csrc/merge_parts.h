// The merge of split-context attention results, made by the product that consumes them.
#pragma once
#include "common.h"

// A given as the unmerged partial results of split-context attention (attention_rows.hip,
// attention_decode.hip): acc [M, heads, parts, d], m and l [M, heads, parts], float32.  Row m, column
// head * d + e of A is sum_p acc_p[e] exp(m_p - max m) / sum_p l_p exp(m_p - max m) over the parts that
// hold keys of the row: the merge of attn_rows_merge_kernel, made while A is staged.
struct UnmergedA {
  const float* acc;
  const float* m;
  const float* l;
  const int* positions;                                    // [M]: a row's context is its position + 1
  int heads, d, parts, P, window;
  const int* part_keys;                                    // null, or where the keys of a part stand (P is not used then)
};
// P == 0 in a launch: the keys of a part stand behind the partial results (attention_decode.hip's plan).
__host__ __device__ inline const int* planned_keys(const float* l, size_t cells, int P) {
  return P ? nullptr : reinterpret_cast<const int*>(l + cells);
}

// The first AT_ONCE parts of E merged values: all their loads, which wait for nothing that stands in memory (without a window the
// parts begin at 0; which of them hold keys of the row is only looked at when they are used).
template <int E, int AT_ONCE>
struct MergeParts {
  float m[AT_ONCE], l[AT_ONCE], acc[AT_ONCE][E];
  int first, position;                                     // the first part that holds keys of the row; the row's position
  // Here they are needed (a load whose use stands under a condition is otherwise moved down to it).
  __device__ __forceinline__ void arrived() {
    asm volatile("" : "+v"(first), "+v"(position));
#pragma unroll
    for (int j = 0; j < AT_ONCE; ++j) {
      asm volatile("" : "+v"(m[j]), "+v"(l[j]));
#pragma unroll
      for (int i = 0; i < E; ++i) asm volatile("" : "+v"(acc[j][i]));
    }
  }
};
__device__ __forceinline__ int merge_part_keys(const UnmergedA& u) { return u.part_keys ? *u.part_keys : u.P; }
template <int E, int AT_ONCE>
__device__ __forceinline__ void merge_load(const UnmergedA& u, size_t cell0, int e, int p0, int most, MergeParts<E, AT_ONCE>& to) {
#pragma unroll
  for (int j = 0; j < AT_ONCE; ++j) {
    const int p = min(p0 + j, most);
    to.m[j] = u.m[cell0 + p];
    to.l[j] = u.l[cell0 + p];
    const float* from = u.acc + (cell0 + p) * u.d + e;
    if constexpr (E == 8) {
      ld8(from, to.acc[j]);
    } else {
      const float4 v = *reinterpret_cast<const float4*>(from);
      to.acc[j][0] = v.x; to.acc[j][1] = v.y; to.acc[j][2] = v.z; to.acc[j][3] = v.w;
    }
  }
}
template <int E, int AT_ONCE>
__device__ __forceinline__ void merge_ask(const UnmergedA& u, int P, int m, int k, MergeParts<E, AT_ONCE>& parts) {
  const int head = k / u.d;
  parts.position = u.positions[m];
  parts.first = u.window > 0 ? max(0, parts.position + 1 - u.window) / P : 0;
  merge_load(u, ((size_t)m * u.heads + head) * u.parts, k - head * u.d, parts.first, u.parts - 1, parts);
}
// E (4 or 8) merged values of row m starting at column k (all of one head: d % E == 0), float32, from what merge_ask loaded
// (P: merge_part_keys, read once by the caller).
// AT_ONCE: parts whose loads are in flight together (E * AT_ONCE registers).
template <int E, int AT_ONCE>
__device__ __forceinline__ void merge_finish(const UnmergedA& u, int P, int m, int k, MergeParts<E, AT_ONCE>& part, float (&out)[E]) {
  const int head = k / u.d, e = k - head * u.d;
  const int first = part.first, last = part.position / P;
  const size_t cell0 = ((size_t)m * u.heads + head) * u.parts;
  // AT_ONCE parts at a time, all their loads first: a loop that waits for memory once per part would cost more
  // than the merge kernel it replaces.  The first parts' sums and values are asked for together with their
  // maxima (they do not depend on the largest maximum, only their use does): one wait for up to AT_ONCE parts.
  float top = -INFINITY;
#pragma unroll
  for (int j = 0; j < AT_ONCE; ++j)
    if (first + j <= last) top = fmaxf(top, part.m[j]);
  for (int p0 = first + AT_ONCE; p0 <= last; p0 += 16) {    // the other parts' maxima, sixteen loads at a time
    float more[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) more[j] = u.m[cell0 + min(p0 + j, last)];
#pragma unroll
    for (int j = 0; j < 16; ++j) top = fmaxf(top, more[j]);
  }
  float denom = 0.f, numer[E];
#pragma unroll
  for (int i = 0; i < E; ++i) numer[i] = 0.f;
  for (int p0 = first; p0 <= last; p0 += AT_ONCE) {
    if (p0 != first) merge_load(u, cell0, e, p0, last, part);
#pragma unroll
    for (int j = 0; j < AT_ONCE; ++j) {                     // the order and the arithmetic of the merge kernel
      if (p0 + j <= last) {
        const float f = expf(part.m[j] - top);
        denom += part.l[j] * f;
#pragma unroll
        for (int i = 0; i < E; ++i) numer[i] += part.acc[j][i] * f;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < E; ++i) out[i] = numer[i] / denom;
}
// The same in one piece, the row's position first and no part past its last one: where nothing else is asked for in between that is mostly
// ahead of merge_ask and merge_finish one behind the other, though it is two trips (float32, us so / those: 16 rows of 896 x 896, 2 parts
// 16.2 / 16.8, 4 of 2,560 x 4,096 13.1 / 13.6; bfloat16: launch_lines in gemm_bf16.hip).
// AT_ONCE: parts whose loads are in flight together (E * AT_ONCE registers).
template <int E, int AT_ONCE = 4>
__device__ __forceinline__ void merged_values(const UnmergedA& u, int m, int k, float (&out)[E]) {
  const int head = k / u.d, e = k - head * u.d;
  const int ctx = u.positions[m] + 1;
  const int lo = u.window > 0 ? max(0, ctx - u.window) : 0;
  const int P = u.part_keys ? *u.part_keys : u.P;
  const int first = lo / P, last = (ctx - 1) / P;
  const size_t cell0 = ((size_t)m * u.heads + head) * u.parts;
  auto load = [&](const float* p, float (&to)[E]) {
    if constexpr (E == 8) {
      ld8(p, to);
    } else {
      const float4 v = *reinterpret_cast<const float4*>(p);
      to[0] = v.x; to[1] = v.y; to[2] = v.z; to[3] = v.w;
    }
  };
  // AT_ONCE parts at a time, all their loads first: a loop that waits for memory once per part would cost more
  // than the merge kernel it replaces.  The first parts' sums and values are asked for together with their
  // maxima (they do not depend on the largest maximum, only their use does): one wait for up to AT_ONCE parts.
  float mv[AT_ONCE], lv[AT_ONCE], part[AT_ONCE][E];
#pragma unroll
  for (int j = 0; j < AT_ONCE; ++j) {
    const int p = min(first + j, last);
    mv[j] = u.m[cell0 + p];
    lv[j] = u.l[cell0 + p];
    load(u.acc + (cell0 + p) * u.d + e, part[j]);
  }
  float top = -INFINITY;
#pragma unroll
  for (int j = 0; j < AT_ONCE; ++j) top = fmaxf(top, mv[j]);
  for (int p0 = first + AT_ONCE; p0 <= last; p0 += 16) {    // the other parts' maxima, sixteen loads at a time
    float more[16];
#pragma unroll
    for (int j = 0; j < 16; ++j) more[j] = u.m[cell0 + min(p0 + j, last)];
#pragma unroll
    for (int j = 0; j < 16; ++j) top = fmaxf(top, more[j]);
  }
  float denom = 0.f, numer[E];
#pragma unroll
  for (int i = 0; i < E; ++i) numer[i] = 0.f;
  for (int p0 = first; p0 <= last; p0 += AT_ONCE) {
    if (p0 != first) {
#pragma unroll
      for (int j = 0; j < AT_ONCE; ++j) {
        const int p = min(p0 + j, last);
        mv[j] = u.m[cell0 + p];
        lv[j] = u.l[cell0 + p];
        load(u.acc + (cell0 + p) * u.d + e, part[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < AT_ONCE; ++j) {                     // the order and the arithmetic of the merge kernel
      if (p0 + j <= last) {
        const float f = expf(mv[j] - top);
        denom += lv[j] * f;
#pragma unroll
        for (int i = 0; i < E; ++i) numer[i] += part[j][i] * f;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < E; ++i) out[i] = numer[i] / denom;
}
