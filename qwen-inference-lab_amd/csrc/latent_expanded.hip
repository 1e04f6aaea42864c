// Latent attention of whole prompts with the heads' keys and values expanded, bfloat16: for steps whose sequences all begin
// at their first token, so that the step's own rows are all the keys there are.  The latents c of the step are multiplied
// out once, K_h = W_uk,h c and V_h = W_uv,h c (two products of the step's rows), and
//     score(h, i, j) = scale * (q_h,i . k_h,j + qr_h,i . kr_j),   out_h,i = sum_j p(h, i, j) v_h,j,   a sink in the divisor,
// runs over 192 + 128 numbers a pair of rows and head where attention over the latents themselves
// (latent_attention_mfma.hip) runs over 576 + 512: bound by the matrix cores and the instructions beside them, prompts of
// 1,777 and 1,267 rows of 16 heads take 62 us a layer and 28 for the two products, and took 398 there with two products per
// head around it besides (a step of 6 layers, 3 of them these: 4.94 -> 3.42 ms; one prompt of 4,001 rows 7.95 -> 4.47).
// Logits of such a step lie 1.08e-2 from float64 (eight inputs on average), over the latents 1.13e-2.
//
// A block is 4 waves of 32 rows each of one head, which share its staged keys; a wave's rows are one tile of
// v_mfma_f32_32x32x16_bf16, as in attention_prompt.hip, whose score layout this is (S^T = K Q^T, 24 products a tile of 64
// keys, softmax in registers, O^T += V^T P^T, 16 products).  Keys and values lie packed, so there are no pages: a wave's
// loads put 1 KB each straight into LDS, and which piece a lane loads makes the layout there:
//   K  [64 rows][16 pieces of 16 bytes]: a load is 4 rows, piece p of row r holds the dims 8 (p ^ (r & 15)) ..;
//   Kr [64 rows][8 pieces]: a load is 8 rows, piece p of row r holds the dims 8 (p ^ (r & 7)) ..;
//   V^T [128 dims][8 pieces of 8 keys]: V comes transposed from its product (the weight is the left operand), a load is
//       8 dims of all 64 keys, whole lines; piece p of dim d holds the keys 8 (p ^ (d & 7)) ..
// Tiles begin at multiples of 64 packed rows, whatever row a sequence begins at: the first and the last tile of a sequence
// hold rows of others, whose scores are masked and whose values are zeroed in LDS (anything might stand there).
// Two tiles in LDS (80 KB: two blocks a CU), one barrier a tile, the next tile's loads sent between the score products.
// Blocks of one head go to one XCD (the head numbers the grid fastest), whose L2 then holds its keys; the row tiles that
// see the most keys come first.
#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

#define EXP_DIM 128                                        // of a head's unrotated keys and queries, and of its values
#define EXP_ROT 64
#define EXP_BK 64
#define EXP_ROWS 128                                       // rows of a block
#define EXP_K_BYTES (EXP_BK * EXP_DIM * 2)
#define EXP_R_BYTES (EXP_BK * EXP_ROT * 2)
#define EXP_TILE_BYTES (2 * EXP_K_BYTES + EXP_R_BYTES)     // K, Kr, V^T: 40 KB

// The key that row r of a score tile holds: a lane's 16 scores of 32 keys are then 8 consecutive keys twice.
__device__ __forceinline__ int expanded_key(int r) { return (r & ~15) + ((r >> 3) & 1) * 4 + ((r >> 2) & 1) * 8 + (r & 3); }

__global__ void __launch_bounds__(4 * QIL_WAVE, 2)
latent_expanded_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k, const bf16_t* __restrict__ kr,
                       const bf16_t* __restrict__ vt, int v_stride, const int* __restrict__ cu_seqlens,
                       const float* __restrict__ freq, const float* __restrict__ sinks, const float* __restrict__ gate,
                       bf16_t* __restrict__ out, int heads, int tiles_x, float scale) {
  constexpr int KF = EXP_DIM / 16, RF = EXP_ROT / 16, QF = KF + RF, VTILES = EXP_DIM / 32;
  extern __shared__ __align__(1024) unsigned char lds[];
  const int id = blockIdx.x, head = id % heads, place = id / heads;
  const int seq = place / tiles_x, across = tiles_x - 1 - place % tiles_x;
  const int begin = cu_seqlens[seq], end = cu_seqlens[seq + 1];
  const int row0 = begin + across * EXP_ROWS;              // rows and keys are numbered through the packed step
  if (row0 >= end) return;
  const int lane = threadIdx.x & (QIL_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / QIL_WAVE);
  const int l32 = lane & 31, half = lane >> 5;
  const int wave_row0 = row0 + 32 * wave, my_row = wave_row0 + l32;
  const bool row_valid = my_row < end;
  const int wave_last = min(end, wave_row0 + 32) - 1;      // no key beyond it is visible to this wave
  const int key_end = min(end, row0 + EXP_ROWS);           // nor beyond this to the block
  const int first_tile = begin / EXP_BK * EXP_BK;

  // the wave's queries: B operand, row l32, dims 16 ks + 8 half ..; the rotated part is turned here (elements i and
  // i + 32 of it are fragments KF + i / 16 and KF + 2 + i / 16 of the same lane)
  bf16x8 qw[QF];
  {
    const bf16_t* from = q + ((size_t)(row_valid ? my_row : row0) * heads + head) * (EXP_DIM + EXP_ROT) + half * 8;
#pragma unroll
    for (int ks = 0; ks < KF; ++ks) qw[ks] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(from + ks * 16));
    const float position = (float)(my_row - begin);
#pragma unroll
    for (int i = 0; i < RF / 2; ++i) {
      float u[8], v[8], turned_u[8], turned_v[8];
      ld8(from + EXP_DIM + i * 16, u);
      ld8(from + EXP_DIM + (i + RF / 2) * 16, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float sn, cs;
        sincosf(position * freq[i * 16 + half * 8 + e], &sn, &cs);
        turned_u[e] = u[e] * cs - v[e] * sn;
        turned_v[e] = v[e] * cs + u[e] * sn;
      }
      auto packed = [](const float (&x)[8]) {
        return __builtin_bit_cast(bf16x8, make_uint4(pack_bf16(x[0], x[1]), pack_bf16(x[2], x[3]), pack_bf16(x[4], x[5]), pack_bf16(x[6], x[7])));
      };
      qw[KF + i] = packed(turned_u);
      qw[KF + RF / 2 + i] = packed(turned_v);
    }
  }
  float row_m = -INFINITY, row_l = 0.f;
  f32x16 ow[VTILES];
#pragma unroll
  for (int t = 0; t < VTILES; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) ow[t][i] = 0.f;

  // ---- loads of a tile: 16 of K (rows 4 j ..), 8 of Kr (rows 8 j ..), 16 of V^T (dims 8 j ..), a quarter of each a wave
  constexpr int LOADS = 10;
  auto load = [&](int i, int k0, unsigned char* to) __attribute__((always_inline)) {
    const char* from;
    unsigned char* at;
    if (i < 4) {
      const int j = 4 * i + wave, r = 4 * j + (lane >> 4);
      from = reinterpret_cast<const char*>(k + ((size_t)(k0 + expanded_key(r)) * heads + head) * EXP_DIM) + (((lane & 15) ^ (r & 15)) << 4);
      at = to + j * 1024;
    } else if (i < 6) {
      const int j = 4 * (i - 4) + wave, r = 8 * j + (lane >> 3);
      from = reinterpret_cast<const char*>(kr + (size_t)(k0 + expanded_key(r)) * EXP_ROT) + (((lane & 7) ^ (r & 7)) << 4);
      at = to + EXP_K_BYTES + j * 1024;
    } else {
      const int j = 4 * (i - 6) + wave, d = 8 * j + (lane >> 3);
      from = reinterpret_cast<const char*>(vt + ((size_t)head * EXP_DIM + d) * v_stride + k0) + (((lane & 7) ^ (d & 7)) << 4);
      at = to + EXP_K_BYTES + EXP_R_BYTES + j * 1024;
    }
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)from,
                                     (__attribute__((address_space(3))) void*)at, 16, 0, 0);
  };
  // values of keys outside [begin, end) of the tile at `tile` become zero
  auto zero_values = [&](int k0, unsigned char* tile) {
    for (int idx = threadIdx.x; idx < EXP_DIM * 8; idx += 4 * QIL_WAVE) {
      const int d = idx >> 3, key = k0 + (((idx & 7) ^ (d & 7)) << 3);
      if (key >= begin && key + 8 <= end) continue;
      uint4* cell = reinterpret_cast<uint4*>(tile + EXP_K_BYTES + EXP_R_BYTES) + idx;
      const uint4 raw = *cell;
      uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (key + e < begin || key + e >= end) w[e >> 1] &= (e & 1) ? 0x0000ffffu : 0xffff0000u;
      *cell = make_uint4(w[0], w[1], w[2], w[3]);
    }
  };

  const float c = scale * 1.44269504088896f;               // p = exp2((s - m) c)
  auto attend = [&](int k0, const unsigned char* tile, unsigned char* next, bool masked, bool more) __attribute__((always_inline)) {
    auto k_fragment = [&](int kt, int ks) __attribute__((always_inline)) {
      const int r = 32 * kt + l32;
      const unsigned char* at = ks < KF ? tile + r * (EXP_DIM * 2) + (((2 * ks + half) ^ (l32 & 15)) << 4)
                                        : tile + EXP_K_BYTES + r * (EXP_ROT * 2) + (((2 * (ks - KF) + half) ^ (l32 & 7)) << 4);
      return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(at));
    };
    constexpr int AHEAD = 2;
    bf16x8 ka[QF][2];
#pragma unroll
    for (int ks = 0; ks < AHEAD; ++ks)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) ka[ks][kt] = k_fragment(kt, ks);
    f32x16 s[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[kt][i] = 0.f;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < QF; ++ks) {
      if (ks + AHEAD < QF) {
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) ka[ks + AHEAD][kt] = k_fragment(kt, ks + AHEAD);
      }
      s[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[ks][0], qw[ks], s[0], 0, 0, 0);
      if (ks < LOADS && more) load(ks, k0 + EXP_BK, next);
      s[1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[ks][1], qw[ks], s[1], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    if (masked) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int key = k0 + 32 * kt + 16 * (i >> 3) + 8 * half + (i & 7);
          s[kt][i] = key >= begin && key <= my_row ? s[kt][i] : -INFINITY;
        }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[kt][i]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, QIL_WAVE));
    // the exponents' reference moves (to the maximum) only if the maximum is 2^8 beyond it, or there was none
    const bool moves = (mx - row_m) * c > 8.f || (row_m == -INFINITY && mx != -INFINITY);
    const float m_new = moves ? mx : row_m;
    const float base = (m_new == -INFINITY) ? 0.f : m_new;
    const float shift = -base * c;
    float alpha = 1.f;
    if (__builtin_amdgcn_ballot_w64(moves) != 0) {
      alpha = moves ? __builtin_amdgcn_exp2f(fmaf(row_m, c, shift)) : 1.f;
#pragma unroll
      for (int t = 0; t < VTILES; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) ow[t][i] *= alpha;
    }
    row_m = m_new;
    float psum = 0.f;
    bf16x8 pb[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      uint32_t packed[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float p0 = __builtin_amdgcn_exp2f(fmaf(s[u >> 1][8 * (u & 1) + 2 * e], c, shift));
        const float p1 = __builtin_amdgcn_exp2f(fmaf(s[u >> 1][8 * (u & 1) + 2 * e + 1], c, shift));
        psum += p0;
        psum += p1;
        packed[e] = pack_bf16(p0, p1);
      }
      pb[u] = __builtin_bit_cast(bf16x8, make_uint4(packed[0], packed[1], packed[2], packed[3]));
    }
    row_l = row_l * alpha + psum;
    asm volatile("" : "+v"(row_l));                        // summed here, not after the products below
    auto v_fragment = [&](int u, int t) __attribute__((always_inline)) {
      const unsigned char* at = tile + EXP_K_BYTES + EXP_R_BYTES + (32 * t + l32) * (EXP_BK * 2) + (((2 * u + half) ^ (l32 & 7)) << 4);
      return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(at));
    };
    bf16x8 va[4][VTILES];
#pragma unroll
    for (int t = 0; t < VTILES; ++t) va[0][t] = v_fragment(0, t);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      if (u + 1 < 4) {
#pragma unroll
        for (int t = 0; t < VTILES; ++t) va[u + 1][t] = v_fragment(u + 1, t);
      }
#pragma unroll
      for (int t = 0; t < VTILES; ++t) ow[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va[u][t], pb[u], ow[t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

#pragma unroll
  for (int i = 0; i < LOADS; ++i) load(i, first_tile, lds);
  int buffer = 0;
  for (int k0 = first_tile; k0 < key_end; k0 += EXP_BK) {
    unsigned char* tile = lds + buffer * EXP_TILE_BYTES;
    unsigned char* next = lds + (buffer ^ 1) * EXP_TILE_BYTES;
    const bool more = k0 + EXP_BK < key_end;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");       // this wave's loads of the tile have landed
    __syncthreads();                                       // everyone's have, and everyone is done with the tile before
    if (k0 < begin || k0 + EXP_BK > end) {
      zero_values(k0, tile);
      __syncthreads();
    }
    if (wave_row0 < end && k0 <= wave_last) {
      attend(k0, tile, next, k0 < begin || k0 + EXP_BK - 1 > wave_row0, more);
    } else if (more) {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) load(i, k0 + EXP_BK, next);
    }
    buffer ^= 1;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  const float total = row_l + __shfl_xor(row_l, 32, QIL_WAVE);
  if (!row_valid) return;
  float inv = sinks ? sink_reciprocal(total, row_m * scale, sinks[head]) : 1.f / total;
  if (gate) inv *= gate[(size_t)my_row * heads + head];
  bf16_t* to = out + ((size_t)my_row * heads + head) * EXP_DIM;
#pragma unroll
  for (int t = 0; t < VTILES; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j)                            // dims 32 t + 8 j + 4 half + e, e < 4
      *reinterpret_cast<uint2*>(to + 32 * t + 8 * j + 4 * half) =
          make_uint2(pack_bf16(ow[t][4 * j] * inv, ow[t][4 * j + 1] * inv), pack_bf16(ow[t][4 * j + 2] * inv, ow[t][4 * j + 3] * inv));
}

extern "C" {

// 1 if the kernel takes these sizes.
int qil_latent_expanded_takes(int dim, int rot, int vdim) { return dim == EXP_DIM && rot == EXP_ROT && vdim == EXP_DIM; }

// q [rows, heads, 192] (a head's unrotated part first, the rotated one not yet turned), k [padded, heads, 128], kr [padded, 64]
// (turned), vt [heads, 128, padded]: `padded` is rows up to the next multiple of 64, and the rows beyond `rows` are read
// but never used.  Sequences begin at position 0; row cu_seqlens[s] + i of sequence s sees its rows up to itself.  freq: the
// rotation's 32 frequencies.  sinks: null, or float32 [heads].  gate: null, or float32 [rows, heads], a factor on the results.
// out [rows, heads, 128].
int qil_latent_expanded(const void* q, const void* k, const void* kr, const void* vt, int padded, const int* cu_seqlens,
                        const float* freq, const float* sinks, const float* gate, void* out, int n_seqs, int max_query,
                        int heads, float scale, hipStream_t s) {
  if (n_seqs == 0 || max_query == 0) return 0;
  const int tiles_x = (max_query + EXP_ROWS - 1) / EXP_ROWS;
  if (padded % EXP_BK || heads < 1 || (long)tiles_x * n_seqs * heads > (1L << 30) ||
      (((uintptr_t)q | (uintptr_t)k | (uintptr_t)kr | (uintptr_t)vt | (uintptr_t)out) % 16))
    return -1;
  static bool granted = false;
  if (!granted) {
    hipError_t e = hipFuncSetAttribute((const void*)latent_expanded_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 2 * EXP_TILE_BYTES);
    if (e != hipSuccess) return (int)e;
    granted = true;
  }
  hipLaunchKernelGGL(latent_expanded_kernel, dim3(tiles_x * n_seqs * heads), dim3(4 * QIL_WAVE), 2 * EXP_TILE_BYTES, s,
                     (const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)kr, (const bf16_t*)vt, padded, cu_seqlens, freq, sinks,
                     gate, (bf16_t*)out, heads, tiles_x, scale);
  QIL_RETURN_LAUNCH_STATUS();
}

}  // extern "C"
