// True float32 matrix product for the 32-bit path: C[M, N] = A[M, K] W[N, K]^T (+ bias[N]).
//
// Many rows: inputs, products and sums are IEEE float32 FMA on the vector units, no split of K
// across threads, so every element of C is one thread's sequential sum over k and does not depend
// on M, on the row's place in the batch or on the tile it falls into.  Few rows: see the streaming
// kernel below (float32 matrix-core instruction, still no reduced-precision input).  Both operands
// have K contiguous (nn.Linear layout, qil/model.py:32-40).  The tiled kernel: 64 x 64 x 16 tiles in
// LDS, 256 threads, 4 x 4 outputs a thread.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "merge_parts.h"

#define SG_BM 64
#define SG_BN 64
#define SG_BK 16
#define SG_PAD 4

template <bool VEC>
__global__ void __launch_bounds__(256)
sgemm_nt_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                float* __restrict__ C, int M, int N, int K) {
  __shared__ float As[SG_BK][SG_BM + SG_PAD];
  __shared__ float Ws[SG_BK][SG_BN + SG_PAD];
  const int tid = threadIdx.x;
  const int m0 = blockIdx.y * SG_BM, n0 = blockIdx.x * SG_BN;
  const int load_row = tid >> 2, load_k = (tid & 3) * 4;      // 64 rows x 4 quads of k
  const int ty = tid >> 4, tx = tid & 15;

  float acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

  for (int k0 = 0; k0 < K; k0 += SG_BK) {
    float a[4], w[4];
    const int am = m0 + load_row, wn = n0 + load_row, kk = k0 + load_k;
    if (VEC && am < M && kk + 3 < K) {
      const float4 v = *reinterpret_cast<const float4*>(A + (size_t)am * K + kk);
      a[0] = v.x; a[1] = v.y; a[2] = v.z; a[3] = v.w;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) a[i] = (am < M && kk + i < K) ? A[(size_t)am * K + kk + i] : 0.f;
    }
    if (VEC && wn < N && kk + 3 < K) {
      const float4 v = *reinterpret_cast<const float4*>(W + (size_t)wn * K + kk);
      w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = (wn < N && kk + i < K) ? W[(size_t)wn * K + kk + i] : 0.f;
    }
    __syncthreads();                       // previous tile fully consumed
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      As[load_k + i][load_row] = a[i];
      Ws[load_k + i][load_row] = w[i];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < SG_BK; ++k) {
      float av[4], wv[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) av[i] = As[k][ty * 4 + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) wv[j] = Ws[k][tx * 4 + j];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(av[i], wv[j], acc[i][j]);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n < N) C[(size_t)m * N + n] = acc[i][j] + (bias ? bias[n] : 0.f);
    }
  }
}

// Few rows (decode): one wave per output column, lanes stride over K; each (m, n) is still a fixed
// order sum: lane partials in k order, then the wave's butterfly.
#define SV_ROWS 8
__global__ void __launch_bounds__(256)
sgemv_rows_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                  float* __restrict__ C, int M, int N, int K, int m0) {
  const int lane = threadIdx.x & (QIL_WAVE - 1);
  const int n = blockIdx.x * (blockDim.x / QIL_WAVE) + threadIdx.x / QIL_WAVE;
  if (n >= N) return;
  const float* w = W + (size_t)n * K;
  float acc[SV_ROWS];
#pragma unroll
  for (int r = 0; r < SV_ROWS; ++r) acc[r] = 0.f;
  const int rows = min(SV_ROWS, M - m0);
  for (int k = lane; k < K; k += QIL_WAVE) {
    const float wv = w[k];
#pragma unroll
    for (int r = 0; r < SV_ROWS; ++r)
      if (r < rows) acc[r] = fmaf(A[(size_t)(m0 + r) * K + k], wv, acc[r]);
  }
#pragma unroll
  for (int r = 0; r < SV_ROWS; ++r) {
    const float total = wave_sum(acc[r]);
    if (lane == 0 && r < rows) C[(size_t)(m0 + r) * N + n] = total + (bias ? bias[n] : 0.f);
  }
}

// Few rows (decode, up to 64), K % 4 == 0: the product is bound by streaming W once, so it is shaped like the
// bfloat16 streaming kernel (gemm_bf16.hip): a block owns 128 columns (8 waves x 16) and one of
// `splits` ranges of K, stages its slice of A in LDS, and every wave streams its 16 rows of W from
// global memory straight into v_mfma_f32_16x16x4_f32 operands: float32 inputs, float32 products and
// sums on the matrix cores (no reduced-precision mode exists for this instruction).  A lane's
// float4 of W (row r, columns 4 kb .. 4 kb + 3 of a 16-column step) feeds four products, A's float4
// from LDS being laid out the same way.  With splits > 1 the block writes a partial result
// C[split, M, N] that the consuming kernel adds in split order.
typedef float f32x4v __attribute__((ext_vector_type(4)));
#define SF_WAVES 8
#define SF_PAD 4
#define SF_MOST_ROWS 64                                    // rows up to which the product streams W through the matrix cores

template <int MT, int UNROLL>
__global__ void __launch_bounds__(SF_WAVES * QIL_WAVE)
gemm_f32_stream_kernel(const float* __restrict__ A, const float* __restrict__ W, const float* __restrict__ bias,
                       float* __restrict__ C, int M, int N, int K, int steps_per_split, int chunk) {
  extern __shared__ __align__(16) float a_lds[];           // [16 MT][chunk + pad]
  const int lane = threadIdx.x & (QIL_WAVE - 1), wave = threadIdx.x / QIL_WAVE;
  const int r = lane & 15, kb = lane >> 4;
  const int n0 = (blockIdx.x * SF_WAVES + wave) * 16, m0 = blockIdx.y * 16 * MT, split = blockIdx.z;
  const int row_width = chunk + SF_PAD;
  f32x4v acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = (f32x4v){0.f, 0.f, 0.f, 0.f};
  const int k_begin = split * steps_per_split * 16, k_end = min(K, k_begin + steps_per_split * 16);
  const bool row_live = n0 + r < N;
  const float* w_row = W + (size_t)(row_live ? n0 + r : 0) * K;
  for (int kc = k_begin; kc < k_end; kc += chunk) {
    const int width = min(chunk, k_end - kc);
    __syncthreads();
    for (int idx = threadIdx.x; idx < 16 * MT * (chunk / 4); idx += SF_WAVES * QIL_WAVE) {
      const int m = idx / (chunk / 4), c = (idx - m * (chunk / 4)) * 4;
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      if (c < width && m0 + m < M) v = *reinterpret_cast<const float4*>(A + (size_t)(m0 + m) * K + kc + c);
      *reinterpret_cast<float4*>(a_lds + m * row_width + c) = v;
    }
    __syncthreads();
    const int steps = (width + 15) / 16;
    for (int step = 0; step < steps; step += UNROLL) {
      float4 b[UNROLL];
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        const int k = kc + (step + u) * 16 + kb * 4;
        b[u] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (step + u < steps && row_live && k < k_end) {     // W is read once (one block of rows a launch)
          const qil_u32x4 raw = load_once(w_row + k);
          b[u] = make_float4(__uint_as_float(raw[0]), __uint_as_float(raw[1]), __uint_as_float(raw[2]), __uint_as_float(raw[3]));
        }
      }
#pragma unroll
      for (int u = 0; u < UNROLL; ++u) {
        if (step + u < steps) {
#pragma unroll
          for (int t = 0; t < MT; ++t) {
            const float4 a = *reinterpret_cast<const float4*>(a_lds + (t * 16 + r) * row_width + (step + u) * 16 + kb * 4);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b[u].x, acc[t], 0, 0, 0);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b[u].y, acc[t], 0, 0, 0);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b[u].z, acc[t], 0, 0, 0);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b[u].w, acc[t], 0, 0, 0);
          }
        }
      }
    }
  }
  float* out = C + (size_t)split * M * N;
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = m0 + t * 16 + 4 * kb + i, n = n0 + r;
      if (m < M && n < N) out[(size_t)m * N + n] = acc[t][i] + (bias ? bias[n] : 0.f);
    }
}

// Up to 16 rows, K split into ranges of whole 64-column stages: W read in whole cache lines, as the bfloat16
// whole-line kernel reads it (gemm_bf16.hip).  A load instruction takes 4 rows x 256 contiguous bytes (lane l:
// row 4 u + l / 16, 16-byte piece l % 16), three stages of 16 rows x 64 columns are in flight in registers, and
// a stage passes through a wave-private 4 KB LDS buffer that turns it into the operands of
// v_mfma_f32_16x16x4_f32 (pieces stored at piece ^ row, so that writes and reads spread over all banks; LDS
// operations of one wave complete in program order, so the buffer needs no barrier).  The block's slice of A
// (8 or 16 rows) stays in LDS, its rows unpadded and the 16-byte pieces of row m stored at piece ^ (m % 8) within
// every 128 bytes, so that the 8 rows a read touches lie in different banks (8 rows of 4,096 columns and the
// buffers are 160 KB exactly: the logits of up to 8 rows at 8B sizes run here unsplit).  The fragment-layout kernel above touches half a cache line per row and load and
// reaches about 3 TB/s at 8B layer sizes; this one streams at 4.3 to 5.6.  Always writes partial sums
// C[split, M, N] (one split: the product itself).
#define FL_WAVES 8                                         // waves of a block: 8, or what fl_waves says
#define FL_NARROW_WAVES 4                                  // small products: twice the blocks
#define FL_WIDE_WAVES 16                                   // one such block fills a CU: A's slice is staged once for 256 columns
#define FL_STAGE 64                                        // columns of a stage
#define FL_PAD 4                                           // floats between rows of a stage of A (the 17-to-64-row kernel)
#define FL_DEPTH 3                                         // stages of W in flight per wave
#define FL_LDS_LIMIT (100 * 1024)
#define FL_WIDE_LDS_LIMIT (160 * 1024)

// A given as the gate and up products of a gated feed-forward, left as partial sums: sums [splits][M][2 K] with
// the gate columns first or (interleaved) gate and up columns in turns of 16.  Row m, column k of A is
// silu(gate[m, k]) * up[m, k] with both summed in split order: what silu_mul in elementwise.hip makes (qil/model.py:71).
struct GatedA {
  const float* sums;
  int splits, interleaved;
};

// ASRC: 0 = A as it is, 1 = merged attention parts (UnmergedA), 2 = the activation of a gated feed-forward (GatedA)
// AHEAD (ASRC 1 and 2): W's first requests go out ahead of the operand's arrival (launch_f32_lines).
template <int ASRC, int WAVES, bool AHEAD = false>
__global__ void __launch_bounds__(WAVES * QIL_WAVE)
gemm_f32_lines_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C, int M, int N, int K,
                      int cols_per_split, UnmergedA unmerged, GatedA gated) {
  extern __shared__ __align__(16) float fl_lds[];           // A slice [8 or 16][cols + pad], then the waves' buffers
  const int lane = threadIdx.x & (QIL_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / QIL_WAVE);
  const int r = lane & 15, kb = lane >> 4;
  const int a_rows = M <= 8 ? 8 : 16;                      // rows of A kept (a power of two)
  const int n0 = (blockIdx.x * WAVES + wave) * 16, split = blockIdx.z;
  const int k_begin = split * cols_per_split, stages = cols_per_split / FL_STAGE;
  const int row_width = cols_per_split;
  float* a_lds = fl_lds;
  float* buffer = fl_lds + a_rows * row_width + wave * (16 * FL_STAGE);

  const int load_row = lane >> 4, piece = lane & 15;
  const float* source[4];                                  // rows past N read a valid row and are never stored
  int place[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int row = 4 * u + load_row;
    source[u] = W + (size_t)min(n0 + row, N - 1) * K + k_begin + piece * 4;
    place[u] = row * FL_STAGE + ((piece ^ row) & 15) * 4;
  }
  // every wave walks its K range from a start of its own and wraps around (waves that read the same columns
  // of their rows at the same time load a few memory channels only)
  const int turn = (n0 / 16) % stages;
  auto column = [&](int stage) { const int st = stage + turn; return (st >= stages ? st - stages : st) * FL_STAGE; };
  f32x4v w0[4], w1[4], w2[4];                              // three stages, named so that none is indexed at run time
  auto request = [&](f32x4v (&stage_w)[4], int stage) {
    const int at = column(stage);
#pragma unroll
    for (int u = 0; u < 4; ++u) stage_w[u] = __builtin_bit_cast(f32x4v, load_once(source[u] + at));
  };
  auto request_first = [&]() {
    request(w0, 0);                                         // the host sees to stages >= 3
    request(w1, 1);
    request(w2, 2);
  };
  // A slice first, W's first stages right behind it where that is possible: loads come back in order, so A's arrival is waited for
  // without W's.  (Rows past M stay as they are in LDS: their products are never stored.)
  constexpr int THREADS = WAVES * QIL_WAVE;
  const int pieces = cols_per_split / 4, all = M * pieces;
  if constexpr (ASRC == 0) {
    // straight into LDS, 256 columns of a row an instruction (lane l's 16 bytes land at piece l: it fetches the piece that belongs there)
    for (int c0 = 0; c0 < cols_per_split; c0 += 256)
      if (c0 + lane * 4 < cols_per_split) {
#pragma unroll 4
        for (int m = wave; m < M; m += WAVES)
          __builtin_amdgcn_global_load_lds(
              (const __attribute__((address_space(1))) void*)(A + (size_t)m * K + k_begin + c0 + ((lane ^ (m & 7)) << 2)),
              (__attribute__((address_space(3))) void*)(a_lds + m * row_width + c0), 16, 0, 0);
      }
    request_first();
    __builtin_amdgcn_s_waitcnt(0x07C);                      // vmcnt(12) lgkmcnt(0): see the whole-line kernel in gemm_bf16.hip
    __builtin_amdgcn_s_barrier();
  } else {
    MergeParts<4, 16> parts;                                // (ASRC 1, AHEAD)
    const int P = ASRC == 1 && AHEAD ? merge_part_keys(unmerged) : 0;
    float4 gs[4], us[4];                                    // (ASRC 2: four splits of gate and up)
    const size_t stride = (size_t)M * 2 * K;
    int m, c;
    auto ask_sums = [&](int s0) __attribute__((always_inline)) {
      const int k = k_begin + c;                            // four columns of one tile of 16
      const size_t at = (size_t)m * 2 * K + (gated.interleaved ? (size_t)(k >> 4) * 32 + (k & 15) : (size_t)k);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const size_t from = (size_t)min(s0 + j, gated.splits - 1) * stride + at;
        gs[j] = *reinterpret_cast<const float4*>(gated.sums + from);
        us[j] = *reinterpret_cast<const float4*>(gated.sums + from + (gated.interleaved ? 16 : K));
      }
    };
    auto ask = [&](int idx) __attribute__((always_inline)) {
      m = idx / pieces;
      c = (idx - m * pieces) * 4;
      if constexpr (ASRC == 2) ask_sums(0);
      else if constexpr (AHEAD) merge_ask(unmerged, P, m, k_begin + c, parts);
    };
    auto put = [&]() __attribute__((always_inline)) {
      float4 v;
      if constexpr (ASRC == 1) {
        float merged[4];
        if constexpr (AHEAD) merge_finish(unmerged, P, m, k_begin + c, parts, merged);
        else merged_values<4, WAVES == FL_WIDE_WAVES ? 8 : 16>(unmerged, m, k_begin + c, merged);      // (sixteen parts do not fit the registers of 16 waves)
        v = make_float4(merged[0], merged[1], merged[2], merged[3]);
      } else {
        float4 g = make_float4(0.f, 0.f, 0.f, 0.f), u = g;
        auto add = [&](int s0) __attribute__((always_inline)) {           // in split order
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (s0 + j < gated.splits) {
              g.x += gs[j].x; g.y += gs[j].y; g.z += gs[j].z; g.w += gs[j].w;
              u.x += us[j].x; u.y += us[j].y; u.z += us[j].z; u.w += us[j].w;
            }
        };
        add(0);
        if constexpr (!AHEAD)
          for (int s0 = 4; s0 < gated.splits; s0 += 4) {
            ask_sums(s0);
            add(s0);
          }
        v = make_float4((g.x / (1.f + expf(-g.x))) * u.x, (g.y / (1.f + expf(-g.y))) * u.y,
                        (g.z / (1.f + expf(-g.z))) * u.z, (g.w / (1.f + expf(-g.w))) * u.w);
      }
      *reinterpret_cast<float4*>(a_lds + m * row_width + (c ^ ((m & 7) << 2))) = v;
    };
    if constexpr (AHEAD) {                                  // (a piece a thread, in one turn of loads: launch_f32_lines)
      ask(min((int)threadIdx.x, all - 1));
      __builtin_amdgcn_sched_barrier(0);
      request_first();
      if constexpr (ASRC == 1) {
        parts.arrived();
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          asm volatile("" : "+v"(gs[j].x), "+v"(gs[j].y), "+v"(gs[j].z), "+v"(gs[j].w), "+v"(us[j].x), "+v"(us[j].y), "+v"(us[j].z), "+v"(us[j].w));
      }
      if ((int)threadIdx.x < all) put();
    } else {
      for (int idx = threadIdx.x; idx < all; idx += THREADS) {
        ask(idx);
        put();
      }
      request_first();
    }
    __syncthreads();
  }

  f32x4v acc = {0.f, 0.f, 0.f, 0.f};
  // lanes past the kept rows read the rows again: their products are rows of D that are never stored
  const float* a_row = a_lds + (r & (a_rows - 1)) * row_width;
  const int a_turn = (r & 7) << 2;                          // where the row's pieces lie within 128 bytes
  auto pass = [&](const f32x4v (&stage_w)[4]) {            // registers -> buffer
#pragma unroll
    for (int u = 0; u < 4; ++u) *reinterpret_cast<f32x4v*>(buffer + place[u]) = stage_w[u];
  };
  auto multiply = [&](int stage) {
    const int at = column(stage);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {                        // columns 16 s4 + 4 kb .. + 3 of the stage: four products
      const f32x4v b = *reinterpret_cast<const f32x4v*>(buffer + r * FL_STAGE + (((4 * s4 + kb) ^ r) & 15) * 4);
      const f32x4v a = *reinterpret_cast<const f32x4v*>(a_row + at + ((s4 * 16 + kb * 4) ^ a_turn));
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, acc, 0, 0, 0);
    }
    __builtin_amdgcn_wave_barrier();
  };
  int stage = 0;
  for (; stage + 6 <= stages; stage += 3) {                 // every stage here has a successor three ahead
    pass(w0); request(w0, stage + 3); multiply(stage);
    pass(w1); request(w1, stage + 4); multiply(stage + 1);
    pass(w2); request(w2, stage + 5); multiply(stage + 2);
  }
  const int left = stages - stage;                          // the last three to five stages: requests run out
  pass(w0); if (left > 3) request(w0, stage + 3); multiply(stage);
  pass(w1); if (left > 4) request(w1, stage + 4); multiply(stage + 1);
  pass(w2); multiply(stage + 2);
  if (left > 3) { pass(w0); multiply(stage + 3); }
  if (left > 4) { pass(w1); multiply(stage + 4); }
  float* out = C + (size_t)split * M * N;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = 4 * kb + i, n = n0 + r;
    if (m < M && n < N) out[(size_t)m * N + n] = acc[i];
  }
}

// 17 to 64 rows, K split into ranges of whole stages: the whole-line kernel with A passing through LDS a stage (64
// columns) at a time, in two slots that the block's threads fill in turn from registers loaded three stages ahead,
// as W's are (the scheme of gemm_bf16_chunks_kernel in gemm_bf16.hip).  One barrier a stage.  MT: 16-row tiles of A;
// every W fragment read from the wave's buffer serves MT products.  With 64 rows the matrix cores allow 4.9 TB/s of
// weights (32 products of 16 x 16 x 4 a stage and row tile), about what memory gives.
#define FC_ROW (FL_STAGE + FL_PAD)
#define FC_MOST_ROWS 64

template <int MT>
__global__ void __launch_bounds__(FL_WAVES * QIL_WAVE)
gemm_f32_chunks_kernel(const float* __restrict__ A, const float* __restrict__ W, float* __restrict__ C, int M, int N,
                       int K, int cols_per_split) {
  extern __shared__ __align__(16) float fc_lds[];           // two stages of A [16 MT][64 + pad], then the waves' buffers
  constexpr int A_ROWS = 16 * MT, SLOT = A_ROWS * FC_ROW;
  constexpr int PIECES = A_ROWS * 16 / (FL_WAVES * QIL_WAVE);     // 16-byte pieces of a stage of A per thread
  static_assert(PIECES >= 1, "a stage of A has fewer pieces than the block has threads");
  const int lane = threadIdx.x & (QIL_WAVE - 1), wave = threadIdx.x / QIL_WAVE;
  const int r = lane & 15, kb = lane >> 4;
  const int split = blockIdx.z;
  const int n0 = (blockIdx.x * FL_WAVES + wave) * 16;
  const int k_begin = split * cols_per_split, stages = cols_per_split / FL_STAGE;
  float* buffer = fc_lds + 2 * SLOT + wave * (16 * FL_STAGE);

  const int load_row = lane >> 4, piece = lane & 15;
  const float* source[4];                                  // rows past N read a valid row and are never stored
  int place[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int row = 4 * u + load_row;
    source[u] = W + (size_t)min(n0 + row, N - 1) * K + k_begin + piece * 4;
    place[u] = row * FL_STAGE + ((piece ^ row) & 15) * 4;
  }
  // This thread's pieces of a stage of A.  Rows past M read row M - 1: their products land in rows of the result
  // that are never stored (a load under a condition would make the compiler wait for every load in flight).
  const float* a_source[PIECES];
  int a_place[PIECES];
#pragma unroll
  for (int u = 0; u < PIECES; ++u) {
    const int p = threadIdx.x + u * (FL_WAVES * QIL_WAVE), row = p >> 4, pc = p & 15;
    a_source[u] = A + (size_t)min(row, M - 1) * K + k_begin + pc * 4;
    a_place[u] = row * FC_ROW + pc * 4;
  }
  const int turn = blockIdx.x % stages;
  auto column = [&](int stage) { const int st = stage + turn; return (st >= stages ? st - stages : st) * FL_STAGE; };
  f32x4v w0[4], w1[4], w2[4], a0[PIECES], a1[PIECES], a2[PIECES];
  auto request = [&](f32x4v (&stage_w)[4], int stage) {
    const int at = column(stage);
#pragma unroll
    for (int u = 0; u < 4; ++u) stage_w[u] = __builtin_bit_cast(f32x4v, load_once(source[u] + at));
  };
  auto request_a = [&](f32x4v (&stage_a)[PIECES], int stage) {
    const int at = column(stage);
#pragma unroll
    for (int u = 0; u < PIECES; ++u) stage_a[u] = *reinterpret_cast<const f32x4v*>(a_source[u] + at);
  };
  auto store_a = [&](const f32x4v (&stage_a)[PIECES], int stage) {
    float* slot = fc_lds + (stage & 1) * SLOT;
#pragma unroll
    for (int u = 0; u < PIECES; ++u) *reinterpret_cast<f32x4v*>(slot + a_place[u]) = stage_a[u];
  };
  request_a(a0, 0); request_a(a1, 1); request_a(a2, 2);     // the host sees to stages >= 3
  request(w0, 0); request(w1, 1); request(w2, 2);
  store_a(a0, 0);
  if (3 < stages) request_a(a0, 3);
  __syncthreads();

  f32x4v acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = (f32x4v){0.f, 0.f, 0.f, 0.f};
  auto pass = [&](const f32x4v (&stage_w)[4]) {            // registers -> buffer
#pragma unroll
    for (int u = 0; u < 4; ++u) *reinterpret_cast<f32x4v*>(buffer + place[u]) = stage_w[u];
  };
  auto multiply = [&](int stage) {
    const float* a_row = fc_lds + (stage & 1) * SLOT + r * FC_ROW + kb * 4;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {                        // columns 16 s4 + 4 kb .. + 3 of the stage: four products a tile
      const f32x4v b = *reinterpret_cast<const f32x4v*>(buffer + r * FL_STAGE + (((4 * s4 + kb) ^ r) & 15) * 4);
      f32x4v a[MT];
#pragma unroll
      for (int t = 0; t < MT; ++t) a[t] = *reinterpret_cast<const f32x4v*>(a_row + t * 16 * FC_ROW + s4 * 16);
#pragma unroll
      for (int c = 0; c < 4; ++c)                           // the tiles in turn: a product never waits for the one before it
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[t][c], b[c], acc[t], 0, 0, 0);
    }
    __builtin_amdgcn_wave_barrier();
  };
  // Stage s: its W goes from registers w to the buffer; registers a hold stage s + 1 of A.  `inner`: every request
  // of the stage has a target (a request under a condition, even a uniform one, makes the compiler wait for all
  // loads in flight at the next use of any of them, so the stages that need conditions are apart).
  auto step = [&](int s, f32x4v (&w)[4], f32x4v (&a)[PIECES], auto inner) {
    pass(w);
    if (decltype(inner)::value || s + 3 < stages) request(w, s + 3);
    if (decltype(inner)::value || s + 1 < stages) store_a(a, s + 1);
    if (decltype(inner)::value || s + 4 < stages) request_a(a, s + 4);
    multiply(s);
    __syncthreads();
  };
  int s = 0;
  for (; s + 7 <= stages; s += 3) {
    step(s, w0, a1, std::true_type());
    step(s + 1, w1, a2, std::true_type());
    step(s + 2, w2, a0, std::true_type());
  }
  for (; s + 3 <= stages; s += 3) {
    step(s, w0, a1, std::false_type());
    step(s + 1, w1, a2, std::false_type());
    step(s + 2, w2, a0, std::false_type());
  }
  if (s < stages) step(s, w0, a1, std::false_type());
  if (s + 1 < stages) step(s + 1, w1, a2, std::false_type());
  float* out = C + (size_t)split * M * N;
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = t * 16 + 4 * kb + i, n = n0 + r;
      if (m < M && n < N) out[(size_t)m * N + n] = acc[t][i];
    }
}

static bool fc_takes(int M, int N, int K, int splits) {
  return M > 16 && M <= FC_MOST_ROWS && N >= 1 && splits >= 1 && K % (FL_STAGE * splits) == 0 &&
         K / (FL_STAGE * splits) >= FL_DEPTH;
}

// K splits of that kernel: the most (a power of two up to 8, with at least three stages each) that keep the blocks
// within the 256 CUs (the rule of the bfloat16 kernel of the same shape).
static int fc_splits(int M, int N, int K) {
  if (!fc_takes(M, N, K, 1)) return 0;
  const long tiles = (N + 16 * FL_WAVES - 1) / (16 * FL_WAVES);
  int splits = 1;
  for (int c = 2; c <= 8; c *= 2)
    if (tiles * c <= QIL_CUS && fc_takes(M, N, K, c)) splits = c;
  return splits;
}

template <int MT>
static int launch_f32_chunks(const float* A, const float* W, float* C, int M, int N, int K, int splits, hipStream_t s) {
  const size_t lds = ((size_t)2 * 16 * MT * FC_ROW + (size_t)FL_WAVES * 16 * FL_STAGE) * sizeof(float);
  auto kernel = gemm_f32_chunks_kernel<MT>;
  static size_t granted = 0;                              // per instantiation
  if (lds > 64 * 1024 && lds > granted) {
    hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
    granted = lds;
  }
  dim3 grid((N + 16 * FL_WAVES - 1) / (16 * FL_WAVES), 1, splits);
  hipLaunchKernelGGL(kernel, grid, dim3(FL_WAVES * QIL_WAVE), lds, s, A, W, C, M, N, K, K / splits);
  QIL_RETURN_LAUNCH_STATUS();
}

static size_t fl_lds_bytes(int M, int K, int splits, int waves = FL_WAVES) {
  return ((size_t)(M <= 8 ? 8 : 16) * (K / splits) + (size_t)waves * 16 * FL_STAGE) * sizeof(float);
}

// all_lds: the block may take all of a CU's LDS (a product that must not be split; the plans keep blocks of 8 waves
// to FL_LDS_LIMIT, which the splits they were measured with fit in)
static bool fl_takes(int M, int N, int K, int splits, int waves = FL_WAVES, bool all_lds = false) {
  return M >= 1 && M <= 16 && N >= 1 && splits >= 1 && K % (FL_STAGE * splits) == 0 &&
         K / (FL_STAGE * splits) >= FL_DEPTH &&
         fl_lds_bytes(M, K, splits, waves) <= (waves != FL_WIDE_WAVES && !all_lds ? FL_LDS_LIMIT : FL_WIDE_LDS_LIMIT);
}

// How well the blocks of `splits` splits and `waves` waves fill their rounds of 256 CUs, less 1.5 % a split for what
// the consumer of the partial sums reads; one round of 160 blocks or more counts as full (the rule of the bfloat16
// kernel).  FL_NOT_TAKEN: the kernel does not take the product so (a score of few blocks may be negative).
#define FL_NOT_TAKEN (-1e9)
static double fl_score(int M, int N, int K, int splits, int waves) {
  if (!fl_takes(M, N, K, splits, waves)) return FL_NOT_TAKEN;
  const long blocks = (long)((N + 16 * waves - 1) / (16 * waves)) * splits;
  const long slots = blocks >= 160 && blocks <= QIL_CUS ? blocks : (blocks + QIL_CUS - 1) / QIL_CUS * QIL_CUS;
  return (double)blocks / (double)slots - 0.015 * splits;
}

// Products of at most 16 MB take blocks of 4 waves where those fill more CUs: a CU draws 36 GB/s at most, and 64 or 128 blocks of
// 131 KB each wait for that.  4 rows: 4,096 x 1,024 in four splits 6.7 us with 128 blocks of 8 waves, 5.9 with 256 of 4; 1,024 x
// 2,048 in eight 6.1 with 64, 4.8 with 128; 1,024 x 3,072 5.8 in 16 splits of 8 blocks, 5.2 in 12 of 16 (16 rows 7.0 / 6.4, 6.3 /
// 5.3, 6.0 / 5.8).  Larger ones stream for longer than their blocks start and end: 6,144 x 1,024 level, 6,144 x 4,096 20.9 us in
// 192 blocks of 8 waves, 24.5 in 192 of 4.
#define FL_NARROW_PRODUCT ((size_t)4 << 20)

// The waves of a block for a product in `splits` splits: 8, 4 for small products, or 16 where only such blocks make one full round of the
// chip.  Measured with the gate and up products of 8B layer sizes (403 MB, 8 rows): 768 blocks of 8 waves in 4 splits,
// two a CU and then a third, 81.3 us; 192 blocks of 16 waves in 2 splits, one a CU, 70.3.  Up to 8 rows only: with 16
// rows of A in LDS the down product in 192 wide blocks of 12 splits took 39.2 us against 37.4 in 512 blocks of 8 waves.
static int fl_waves(int M, int N, int K, int splits) {
  if ((size_t)N * K <= FL_NARROW_PRODUCT && fl_score(M, N, K, splits, FL_NARROW_WAVES) > fl_score(M, N, K, splits, FL_WAVES))
    return FL_NARROW_WAVES;
  return M <= 8 && fl_score(M, N, K, splits, FL_WIDE_WAVES) > fl_score(M, N, K, splits, FL_WAVES) ? FL_WIDE_WAVES : FL_WAVES;
}

// The split of K for the whole-line kernel (0: it does not take the product): of the splits it takes (up to 32, with
// the waves that fl_waves gives them), the one with the best score; ties go to fewer splits.
static int fl_splits(int M, int N, int K) {
  int fit = 0;
  double fit_score = 0;
  for (int c = 1; c <= 32; ++c) {
    const double score = fl_score(M, N, K, c, fl_waves(M, N, K, c));
    if (score > FL_NOT_TAKEN && (!fit || score > fit_score)) { fit = c; fit_score = score; }
  }
  return fit;
}

template <int ASRC, int WAVES, bool AHEAD = false>
static int launch_f32_lines_waves(const float* A, UnmergedA unmerged, GatedA gated, const float* W, float* C, int M, int N,
                                  int K, int splits, hipStream_t s) {
  const size_t lds = fl_lds_bytes(M, K, splits, WAVES);
  auto kernel = gemm_f32_lines_kernel<ASRC, WAVES, AHEAD>;
  static size_t granted = 0;                              // per instantiation
  if (lds > 64 * 1024 && lds > granted) {
    hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
    granted = lds;
  }
  dim3 grid((N + 16 * WAVES - 1) / (16 * WAVES), 1, splits);
  hipLaunchKernelGGL(kernel, grid, dim3(WAVES * QIL_WAVE), lds, s, A, W, C, M, N, K, K / splits, unmerged, gated);
  QIL_RETURN_LAUNCH_STATUS();
}

template <int ASRC>
static int launch_f32_lines(const float* A, UnmergedA unmerged, GatedA gated, const float* W, float* C, int M, int N, int K,
                            int splits, hipStream_t s) {
  const int waves = fl_waves(M, N, K, splits);
  if (!fl_takes(M, N, K, splits, waves, splits == 1)) return -1;
  // W ahead of an operand that is made here: in blocks of 4 waves whose threads make one piece each from one turn of loads
  // (4 rows, us behind / ahead: 2,048 x 2,048 behind the merge of 16 parts 7.9 / 6.8, 1,024 x 3,072 behind the activation of four sums 5.9 /
  // 5.0; with A as it is straight into LDS, 16 rows of 4,096 x 1,024 6.3 / 5.7; a step of 28 layers, 4 rows 1,366 -> 1,323).
  if constexpr (ASRC != 0)
    if (waves == FL_NARROW_WAVES && (long)M * (K / splits / 4) <= FL_NARROW_WAVES * QIL_WAVE &&
        (ASRC == 1 ? unmerged.parts <= 16 : gated.splits <= 4))
      return launch_f32_lines_waves<ASRC, FL_NARROW_WAVES, true>(A, unmerged, gated, W, C, M, N, K, splits, s);
  if (waves == FL_NARROW_WAVES) return launch_f32_lines_waves<ASRC, FL_NARROW_WAVES>(A, unmerged, gated, W, C, M, N, K, splits, s);
  return waves == FL_WAVES ? launch_f32_lines_waves<ASRC, FL_WAVES>(A, unmerged, gated, W, C, M, N, K, splits, s)
                           : launch_f32_lines_waves<ASRC, FL_WIDE_WAVES>(A, unmerged, gated, W, C, M, N, K, splits, s);
}

// The whole-line product with the merge of split-context attention results made while A is staged
// (A[M, heads * d] is never written).  workspace: acc [M, heads, parts, d], then m and l [M, heads, parts], float32
// (attention_rows.hip).  C float32 [splits, M, N].
extern "C" int qil_gemm_f32_unmerged_takes(int M, int N, int heads, int d, int splits) {
  return heads >= 1 && d >= 4 && d % 4 == 0 && splits >= 1 && fl_takes(M, N, heads * d, splits, fl_waves(M, N, heads * d, splits));
}

extern "C" int qil_gemm_f32_unmerged(const void* workspace, const int* positions, const void* W, float* C, int M, int N,
                                     int heads, int d, int window, int P, int parts, int splits, hipStream_t s) {
  if (M == 0 || N == 0) return 0;
  if (!qil_gemm_f32_unmerged_takes(M, N, heads, d, splits) || parts < 1 || P < 0 ||
      (((uintptr_t)workspace | (uintptr_t)W) % 16))
    return -1;
  UnmergedA u;
  u.acc = (const float*)workspace;
  u.m = u.acc + (size_t)M * heads * parts * d;
  u.l = u.m + (size_t)M * heads * parts;
  u.positions = positions;
  u.heads = heads; u.d = d; u.parts = parts; u.P = P; u.window = window;
  u.part_keys = planned_keys(u.l, (size_t)M * heads * parts, P);
  return launch_f32_lines<1>(nullptr, u, GatedA(), (const float*)W, C, M, N, heads * d, splits, s);
}

// The whole-line product of the activation of a gated feed-forward, made from the gate and up products' partial
// sums while A is staged: sums float32 [sum_splits, M, 2 K].  C float32 [splits, M, N].
extern "C" int qil_gemm_f32_gated_takes(int M, int N, int K, int interleaved, int splits) {
  return splits >= 1 && (!interleaved || K % 16 == 0) && fl_takes(M, N, K, splits, fl_waves(M, N, K, splits));
}

extern "C" int qil_gemm_f32_gated(const float* sums, int sum_splits, int interleaved, const void* W, float* C, int M, int N,
                                  int K, int splits, hipStream_t s) {
  if (M == 0 || N == 0) return 0;
  if (!qil_gemm_f32_gated_takes(M, N, K, interleaved, splits) || sum_splits < 1 || (((uintptr_t)sums | (uintptr_t)W) % 16))
    return -1;
  GatedA g;
  g.sums = sums; g.splits = sum_splits; g.interleaved = interleaved;
  return launch_f32_lines<2>(nullptr, UnmergedA(), g, (const float*)W, C, M, N, K, splits, s);
}

extern "C" int qil_gemm_f32_mfma_takes(int M, int N, int K, int splits);      // gemm_f32_mfma.hip
extern "C" long qil_gemm_f32_mfma_blocks(int M, int N);
extern "C" int qil_gemm_f32_mfma_splits(int M, int N, int K);
extern "C" int qil_gemm_f32_mfma(const float* A, const float* W, const float* bias, float* C, int M, int N, int K,
                                 int splits, hipStream_t s);

// More than 64 rows: the matrix-core kernel where it takes the sizes (K in whole stages of 32) and is the faster one
// by this count.  A block of the matrix-core kernel runs through its part of K at 3.9 us a stage (2.0 with 128 rows),
// one block a CU; the vector units' kernel takes 0.069 us a column of K however few rows there are and reaches 61 to
// 74 TFLOP/s with many.  Measured at K = 4,096 unsplit: 1,024 x 6,144 in 192 blocks 546 against 755 us, 512 x 6,144 in
// 96 blocks 522 against 420; in two splits 276.
static bool mfma_wanted(int M, int N, int K, int splits) {
  if (M <= SF_MOST_ROWS || !qil_gemm_f32_mfma_takes(M, N, K, splits)) return false;
  const double rounds = (double)((qil_gemm_f32_mfma_blocks(M, N) * splits + QIL_CUS - 1) / QIL_CUS);
  const double matrix = rounds * (K / 32 / splits) * (M <= 128 ? 2.0 : 3.9) + 8.0;
  const double vector = std::max(0.069 * K, 2.0 * ((M + 63) / 64 * 64) * N * (double)K / 66e6);   // 64-row tiles, 61 to 74 TFLOP/s
  return matrix < vector;
}

// Waves of a block of the whole-line kernel for a product of up to 16 rows in `splits` splits (4, 8 or 16; 0: another
// kernel runs it).
extern "C" int qil_gemm_f32_waves(int M, int N, int K, int splits) {
  if (M < 1 || M > 16 || K % 4 || splits < 1) return 0;
  const int waves = fl_waves(M, N, K, splits);
  return fl_takes(M, N, K, splits, waves, splits == 1) && (splits == 1 || splits == fl_splits(M, N, K)) ? waves : 0;
}

// Ways the product will be split over K when partial sums are allowed (1: it is not split).
extern "C" int qil_gemm_f32_splits(int M, int N, int K) {
  if (M > SF_MOST_ROWS) {
    const int sp = qil_gemm_f32_mfma_splits(M, N, K);
    return mfma_wanted(M, N, K, sp) ? sp : 1;
  }
  if (K % 4) return 1;
  if (const int lines = fl_splits(M, N, K)) return lines;
  if (const int chunks = fc_splits(M, N, K)) return chunks;
  const int column_blocks = (N + 127) / 128, steps = (K + 15) / 16;
  int sp = (3 * QIL_CUS + column_blocks - 1) / column_blocks;
  if (sp > 8) sp = 8;
  while (sp > 1 && steps / sp < 16) --sp;
  return sp < 1 ? 1 : sp;
}

// C float32 [splits, M, N] (the value is the sum over the first axis); splits > 1 needs no bias and either M <= 64
// and K % 4 == 0, or the number of splits that qil_gemm_f32_splits gives for more rows.
extern "C" int qil_gemm_f32(const float* A, const float* W, const float* bias, float* C, int M, int N, int K,
                            int splits, hipStream_t s) {
  if (M == 0 || N == 0) return 0;
  if (K < 1 || splits < 1) return -1;
  const bool stream_ok = M <= SF_MOST_ROWS && K % 4 == 0 && (((uintptr_t)A | (uintptr_t)W) % 16 == 0);
  if (M > SF_MOST_ROWS && mfma_wanted(M, N, K, splits) && !(bias && splits > 1) &&
      (((uintptr_t)A | (uintptr_t)W | (uintptr_t)C) % 16) == 0)
    return qil_gemm_f32_mfma(A, W, bias, C, M, N, K, splits, s);
  if (splits > 1 && (!stream_ok || bias)) return -1;
  if (stream_ok && !bias && (splits == 1 || splits == fl_splits(M, N, K)) &&
      fl_takes(M, N, K, splits, fl_waves(M, N, K, splits), splits == 1))
    return launch_f32_lines<0>(A, UnmergedA(), GatedA(), W, C, M, N, K, splits, s);
  if (stream_ok && !bias && fc_takes(M, N, K, splits) && (splits == 1 || splits == fc_splits(M, N, K)))
    return M <= 32 ? launch_f32_chunks<2>(A, W, C, M, N, K, splits, s) : launch_f32_chunks<4>(A, W, C, M, N, K, splits, s);
  if (stream_ok) {
    const int mt = M <= 16 ? 1 : M <= 32 ? 2 : 4;           // 16-row tiles of A a block keeps
    const int steps = (K + 15) / 16, steps_per_split = (steps + splits - 1) / splits;
    int chunk = steps_per_split * 16;
    const int cap = (64 * 1024 / (16 * mt * (int)sizeof(float)) - SF_PAD) / 64 * 64;   // columns per row within 64 KB
    if (chunk > cap) chunk = cap;
    chunk = (chunk + 15) / 16 * 16;
    const size_t lds = (size_t)16 * mt * (chunk + SF_PAD) * sizeof(float);
    dim3 grid((N + 127) / 128, 1, splits);
#define QIL_SF_LAUNCH(MT)                                                                                          \
  hipLaunchKernelGGL((gemm_f32_stream_kernel<MT, 4>), grid, dim3(SF_WAVES * QIL_WAVE), lds, s, A, W, bias, C, M, N, K, \
                     steps_per_split, chunk)
    if (mt == 1) QIL_SF_LAUNCH(1); else if (mt == 2) QIL_SF_LAUNCH(2); else QIL_SF_LAUNCH(4);
#undef QIL_SF_LAUNCH
    QIL_RETURN_LAUNCH_STATUS();
  }
  if (M <= 2 * SV_ROWS) {
    const int waves = 4;
    for (int m0 = 0; m0 < M; m0 += SV_ROWS)
      hipLaunchKernelGGL(sgemv_rows_kernel, dim3((N + waves - 1) / waves), dim3(waves * QIL_WAVE), 0, s, A, W, bias, C,
                         M, N, K, m0);
    QIL_RETURN_LAUNCH_STATUS();
  }
  dim3 grid((N + SG_BN - 1) / SG_BN, (M + SG_BM - 1) / SG_BM);
  const bool vec = (K % 4 == 0) && (((uintptr_t)A | (uintptr_t)W) % 16 == 0);
  if (vec) hipLaunchKernelGGL(sgemm_nt_kernel<true>, grid, dim3(256), 0, s, A, W, bias, C, M, N, K);
  else     hipLaunchKernelGGL(sgemm_nt_kernel<false>, grid, dim3(256), 0, s, A, W, bias, C, M, N, K);
  QIL_RETURN_LAUNCH_STATUS();
}
