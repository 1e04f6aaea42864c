// Shared device helpers for the gfx950 kernels: element types, wave and block reductions.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef uint16_t bf16_t;                       // raw bfloat16 bits

#define QIL_WAVE 64
// Compute units the launch plans are made for (an MI355X; qil_device_info tells what the device has, and the
// Python side warns when it differs: the kernels stay right, their plans fit less well).
#define QIL_CUS 256

// Element type codes of the C interface.
enum { QIL_F32 = 0, QIL_BF16 = 1 };

__device__ __forceinline__ float bf16_to_f32(bf16_t x) { return __uint_as_float(((uint32_t)x) << 16); }

// Round to nearest even; NaN stays NaN (v_cvt_pk_bf16_f32 on gfx950).
typedef __bf16 qil_bf16x2 __attribute__((ext_vector_type(2)));
typedef float qil_f32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  const qil_f32x2 v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, qil_bf16x2));
}
__device__ __forceinline__ bf16_t f32_to_bf16(float f) { return (bf16_t)(pack_bf16(f, 0.f) & 0xffffu); }

// Sixteen bytes that this kernel reads once and no other block reads (weights of a few-row product, keys and values
// of a decode step): the nontemporal hint keeps them from displacing what the caches hold.  A 200 MB read of such
// data reaches 5.5 TB/s with plain loads and 6.8 TB/s with the hint on this part (16 GB: 6.2 against 7.1).
typedef uint32_t qil_u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ qil_u32x4 load_once(const void* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const qil_u32x4*>(p));
}
// The same hint for a load that goes straight into LDS (the instruction's cache-policy bits).
#define QIL_LOAD_ONCE_POLICY 2

// 16 bytes a lane from `from` (the same for the whole wave) + `lane_offset` bytes straight into LDS at `to` + 16 * lane.  A buffer
// load, for loops that read LDS meanwhile: the global form is a flat instruction to the compiler, and with a flat one in flight it
// waits for ALL of a wave's reads of LDS (lgkmcnt(0)) where the oldest are what it needs.
__device__ __forceinline__ void load_to_lds(const void* from, uint32_t lane_offset, void* to) {
  const __amdgpu_buffer_rsrc_t source = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(from), 0, (int)0xffffffffu, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(source, (__attribute__((address_space(3))) void*)to, 16, lane_offset, 0, 0, 0);
}

__device__ __forceinline__ float ld(const float* p) { return *p; }
__device__ __forceinline__ float ld(const bf16_t* p) { return bf16_to_f32(*p); }
__device__ __forceinline__ void st(float* p, float v) { *p = v; }
__device__ __forceinline__ void st(bf16_t* p, float v) { *p = f32_to_bf16(v); }

// A soft cap of attention scores: cap * tanh(score / cap); cap == 0 leaves the score as it is.  The second form
// (the exponential and the reciprocal of the hardware, a few 1e-7 of the cap off) is for the bfloat16 kernels.
__device__ __forceinline__ float soft_cap(float score, float cap) { return cap > 0.f ? cap * tanhf(score / cap) : score; }
__device__ __forceinline__ float soft_cap_fast(float score, float cap, float doubled_log2e_over_cap) {
  const float t = __builtin_amdgcn_exp2f(score * doubled_log2e_over_cap);       // exp(2 score / cap)
  return cap - 2.f * cap * __builtin_amdgcn_rcpf(t + 1.f);                       // cap * (1 - 2 / (t + 1))
}

// A sink in a softmax: one more term exp(sink) in the denominator, with no key and no value.  With the sum l of
// exp(score - m) over the keys, the weights' divisor is l + exp(sink - m); this is its reciprocal, made so that a
// sink far above every score does not overflow.
__device__ __forceinline__ float sink_reciprocal(float l, float m, float sink) {
  if (sink <= m) return 1.f / (l + expf(sink - m));
  const float t = expf(m - sink);
  return t / (l * t + 1.f);
}

// Value after a round trip through T (what the reference's cast to the model dtype does).
template <typename T> __device__ __forceinline__ float round_to(float v);
template <> __device__ __forceinline__ float round_to<float>(float v) { return v; }
template <> __device__ __forceinline__ float round_to<bf16_t>(float v) { return bf16_to_f32(f32_to_bf16(v)); }

// Eight consecutive elements as floats.  `aligned` promises 16-byte (bf16) / 32-byte-pair (f32) alignment.
__device__ __forceinline__ void ld8(const bf16_t* p, float* out) {
  uint4 raw = *reinterpret_cast<const uint4*>(p);
  uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    out[2 * i] = __uint_as_float(w[i] << 16);
    out[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
  }
}
__device__ __forceinline__ void ld8(const float* p, float* out) {
  float4 a = *reinterpret_cast<const float4*>(p);
  float4 b = *reinterpret_cast<const float4*>(p + 4);
  out[0] = a.x; out[1] = a.y; out[2] = a.z; out[3] = a.w;
  out[4] = b.x; out[5] = b.y; out[6] = b.z; out[7] = b.w;
}

// Four consecutive elements as floats, and back (8 bytes of bfloat16, 16 of float32; aligned to that).
__device__ __forceinline__ float4 ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 ld4(const bf16_t* p) {
  const uint2 raw = *reinterpret_cast<const uint2*>(p);
  return make_float4(__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xffff0000u), __uint_as_float(raw.y << 16),
                     __uint_as_float(raw.y & 0xffff0000u));
}
__device__ __forceinline__ void st4(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }
__device__ __forceinline__ void st4(bf16_t* p, float4 v) {
  *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16(v.x, v.y), pack_bf16(v.z, v.w));
}

// A wave's sum and largest value, in the order of a butterfly over 32, 16, 8, 4, 2, 1 lanes, by moves between registers (a shuffle is
// a trip through LDS of some 60 ns, and six of them stood in every norm and every normed product: a
// decode step of 65 kernels 428 -> 422 us, one of 201 1,380 -> 1,366).
template <int CONTROL>
__device__ __forceinline__ float lane_move(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CONTROL, 0xF, 0xF, true));
}
typedef unsigned int qil_u32x2 __attribute__((ext_vector_type(2)));
template <typename F>
__device__ __forceinline__ float wave_combine(float v, F&& with) {
  const unsigned a = __float_as_uint(v);
  const qil_u32x2 halves = __builtin_bit_cast(qil_u32x2, __builtin_amdgcn_permlane32_swap(a, a, false, false));
  v = with(__uint_as_float(halves[0]), __uint_as_float(halves[1]));               // the lanes 32 apart
  const unsigned b = __float_as_uint(v);
  const qil_u32x2 rows = __builtin_bit_cast(qil_u32x2, __builtin_amdgcn_permlane16_swap(b, b, false, false));
  v = with(__uint_as_float(rows[0]), __uint_as_float(rows[1]));                   // 16 apart
  v = with(v, lane_move<0x128>(v));                                               // a row of 16 rotated by 8
  v = with(v, lane_move<0x124>(v));                                               // by 4 (lanes 8 apart agree by now)
  v = with(v, lane_move<0x4E>(v));                                                // quads (2, 3, 0, 1)
  return with(v, lane_move<0xB1>(v));                                             // quads (1, 0, 3, 2)
}
__device__ __forceinline__ float wave_sum(float v) { return wave_combine(v, [](float x, float y) { return x + y; }); }
__device__ __forceinline__ float wave_max(float v) { return wave_combine(v, [](float x, float y) { return fmaxf(x, y); }); }

// Block reductions for blocks of up to 16 waves; `scratch` holds 16 floats of LDS.
// Every thread of the block must call; every thread gets the result.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  const int lane = threadIdx.x & (QIL_WAVE - 1), wave = threadIdx.x / QIL_WAVE;
  const int waves = (blockDim.x + QIL_WAVE - 1) / QIL_WAVE;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = 0.f;
  for (int w = 0; w < waves; ++w) total += scratch[w];      // fixed order
  return total;
}
__device__ __forceinline__ float block_max(float v, float* scratch) {
  const int lane = threadIdx.x & (QIL_WAVE - 1), wave = threadIdx.x / QIL_WAVE;
  const int waves = (blockDim.x + QIL_WAVE - 1) / QIL_WAVE;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float best = scratch[0];
  for (int w = 1; w < waves; ++w) best = fmaxf(best, scratch[w]);
  return best;
}

// Launch epilogue of every C entry point: 0 on success, the HIP error code otherwise.
#define QIL_RETURN_LAUNCH_STATUS() return (int)hipGetLastError()
