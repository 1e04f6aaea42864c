// An operand that is either one array of the model's type or float32 partial sums of a product split over K
// ([splits][rows][columns], added here in split order): what a consumer of ``ops.linear``'s results reads.
#pragma once
#include "common.h"

struct Operand {
  const void* data;
  int code;            // QIL_F32 | QIL_BF16
  int splits;          // float32 only; 1 for a plain array
  size_t stride;       // elements between two splits
};

__device__ __forceinline__ float operand_at(const Operand& x, size_t index) {
  if (x.code == QIL_BF16) return bf16_to_f32(reinterpret_cast<const bf16_t*>(x.data)[index]);
  const float* base = reinterpret_cast<const float*>(x.data) + index;
  float v = 0.f;
  for (int s0 = 0; s0 < x.splits; s0 += 4) {             // four splits' loads in flight; the additions stay in split order
    float part[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) part[k] = s0 + k < x.splits ? base[(size_t)(s0 + k) * x.stride] : 0.f;
#pragma unroll
    for (int k = 0; k < 4; ++k) v += part[k];
  }
  return v;
}
// Four neighbouring elements (index a multiple of 4, the array 16-byte aligned).
__device__ __forceinline__ float4 operand_at4(const Operand& x, size_t index) {
  if (x.code == QIL_BF16) return ld4(reinterpret_cast<const bf16_t*>(x.data) + index);
  const float* base = reinterpret_cast<const float*>(x.data) + index;
  float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int s0 = 0; s0 < x.splits; s0 += 4) {
    float4 part[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      part[k] = s0 + k < x.splits ? ld4(base + (size_t)(s0 + k) * x.stride) : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int k = 0; k < 4; ++k) { v.x += part[k].x; v.y += part[k].y; v.z += part[k].z; v.w += part[k].w; }
  }
  return v;
}

// operand_at4 in two halves: the load of a plain array, and what becomes of it, for a kernel that asks for its operands
// before it takes the first (operand_at4 waits for its own load inside its branch): the gated group norm, 2,048 rows
// 24.8 -> 22.9 us.  Partial sums are not asked for: their loop has four splits in flight.  The residual join, which has
// five operands, gained 2 us at 2,048 rows only where it asked for partial sums too, and then took 8.8 us instead of 7.7
// for 12 rows (twelve splits: a turn of the loop more).
struct AskedOperand { uint32_t bits[4]; };
__device__ __forceinline__ AskedOperand operand_ask4(const Operand& x, size_t index) {
  AskedOperand asked{};
  if (x.code == QIL_BF16) {
    const uint2 q = *reinterpret_cast<const uint2*>(reinterpret_cast<const bf16_t*>(x.data) + index);
    asked.bits[0] = q.x; asked.bits[1] = q.y;
  } else if (x.splits == 1) {
    const uint4 q = *reinterpret_cast<const uint4*>(reinterpret_cast<const float*>(x.data) + index);
    asked.bits[0] = q.x; asked.bits[1] = q.y; asked.bits[2] = q.z; asked.bits[3] = q.w;
  }
  return asked;
}
__device__ __forceinline__ float4 operand_take4(const Operand& x, size_t index, const AskedOperand& asked) {
  if (x.code == QIL_BF16)
    return make_float4(__uint_as_float(asked.bits[0] << 16), __uint_as_float(asked.bits[0] & 0xffff0000u),
                       __uint_as_float(asked.bits[1] << 16), __uint_as_float(asked.bits[1] & 0xffff0000u));
  if (x.splits == 1)
    return make_float4(__uint_as_float(asked.bits[0]), __uint_as_float(asked.bits[1]), __uint_as_float(asked.bits[2]),
                       __uint_as_float(asked.bits[3]));
  return operand_at4(x, index);
}
