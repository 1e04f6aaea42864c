// bfloat16 matrix product on the matrix cores for few rows (decode, selected logit rows):
//   C[M, N] = A[M, K] W[N, K]^T (+ bias[N]),  float32 accumulation.
// Four kernels, all bound by reading W once: `stream` (this comment; any shape, bias, unaligned operands),
// `lines` (up to 16 rows, W in whole cache lines, optional merge of attention parts into A), `chunks`
// (17 to 192 rows, A through LDS in stages) and `gated` (gate and up products with SiLU in the epilogue).
// Both operands have K contiguous (qil/model.py:32-40).  The product is bound by streaming W once
// from HBM; A is small and would be re-read from L2 by every block, so the work is cut into wide,
// short pieces: a block owns 128 * NT rows of W (8 waves, each 16 * NT rows) and ONE of `splits`
// ranges of K.  It stages its slice of A in LDS once, then every wave streams its rows of W from
// global memory straight into v_mfma_f32_16x16x32_bf16 operands, loading UNROLL k steps ahead of
// the first product that uses them.  A's traffic is M / (128 NT) of W's.
//
// With splits > 1 a block writes a float32 partial result C[split, M, N], and the kernel that
// consumes the product (norm, rotary/store, SiLU gate) adds the partials in split order, so
// every sum is made in a fixed order.  With splits == 1 the result may be rounded to bfloat16
// here and take the bias.
//
// Fragment layout of v_mfma_f32_16x16x32_bf16 (wave64): lane l supplies A[l % 16][8 (l / 16) .. +7]
// and B[8 (l / 16) .. +7][l % 16]; it receives D[4 (l / 16) + i][l % 16], i < 4.  A and W rows are
// both loaded with the same k assignment, so only the D layout matters for correctness.
#include <algorithm>
#include <type_traits>

#include "common.h"
#include "gated_act.h"
#include "merge_parts.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void store_out(float* p, float v) { *p = v; }
__device__ __forceinline__ void store_out(bf16_t* p, float v) { *p = f32_to_bf16(v); }

// Eight consecutive bf16 of a row starting at k, zero where the row or k is out of range.  ONCE: the row belongs to W,
// which this kernel reads once (load_once in common.h).
template <bool ALIGNED, bool ONCE = false>
__device__ __forceinline__ uint4 load_frag(const bf16_t* __restrict__ base, int row, int rows, int k, int K) {
  uint4 raw = make_uint4(0, 0, 0, 0);
  if (row < rows && k < K) {
    const bf16_t* p = base + (size_t)row * K + k;
    if (ALIGNED && ONCE) {
      const qil_u32x4 v = load_once(p);
      raw = make_uint4(v[0], v[1], v[2], v[3]);
    } else if (ALIGNED) {
      raw = *reinterpret_cast<const uint4*>(p);
    } else {
      uint32_t w[4] = {0, 0, 0, 0};
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (k + e < K) w[e >> 1] |= (uint32_t)p[e] << ((e & 1) * 16);
      raw = make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
  return raw;
}

#define GEMM_WAVES 8
#define GEMM_LDS_PAD 8          // bf16 elements between rows of the staged A slice

// chunk: k columns of A staged at a time (a multiple of 32); the block's range is walked in chunks.
template <int MT, int NT, int UNROLL, bool ALIGNED, typename OUT>
__global__ void __launch_bounds__(GEMM_WAVES * QIL_WAVE)
gemm_bf16_stream_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, const float* __restrict__ bias,
                        OUT* __restrict__ C, int M, int N, int K, int steps_per_split, int chunk) {
  extern __shared__ __align__(16) bf16_t a_lds[];          // [16 MT][chunk + pad]
  const int lane = threadIdx.x & (QIL_WAVE - 1), wave = threadIdx.x / QIL_WAVE;
  const int r = lane & 15, kb = lane >> 4;
  const int n0 = (blockIdx.x * GEMM_WAVES + wave) * 16 * NT, m0 = blockIdx.y * 16 * MT, split = blockIdx.z;
  const int row_width = chunk + GEMM_LDS_PAD;

  f32x4 acc[MT][NT];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[t][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

  const int k_begin = split * steps_per_split * 32, k_end = min(K, k_begin + steps_per_split * 32);
  // W fragments of the next UNROLL k steps are always in flight: the first group is requested before A
  // is even staged, and each later group before the products of the group in hand.  Two register
  // buffers take turns; the loop is written out in pairs so that each is indexed statically.
  uint4 b0[UNROLL][NT], b1[UNROLL][NT];
  auto request = [&](uint4 (&b)[UNROLL][NT], int k0) {     // k steps starting at column k0
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int k = k0 + u * 32 + kb * 8;
#pragma unroll
      for (int j = 0; j < NT; ++j) b[u][j] = load_frag<ALIGNED, true>(W, n0 + j * 16 + r, N, k < k_end ? k : K, K);
    }
  };
  auto multiply = [&](const uint4 (&b)[UNROLL][NT], int step, int steps) {
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      if (step + u < steps) {
#pragma unroll
        for (int t = 0; t < MT; ++t) {
          const uint4 a = *reinterpret_cast<const uint4*>(a_lds + (t * 16 + r) * row_width + (step + u) * 32 + kb * 8);
#pragma unroll
          for (int j = 0; j < NT; ++j)
            acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                                __builtin_bit_cast(bf16x8, b[u][j]), acc[t][j], 0, 0, 0);
        }
      }
    }
  };
  request(b0, k_begin);
  for (int kc = k_begin; kc < k_end; kc += chunk) {          // chunk is a multiple of 64 * UNROLL columns
    const int width = min(chunk, k_end - kc);               // columns of this chunk (last one may be short)
    __syncthreads();                                        // the previous chunk is consumed
    for (int idx = threadIdx.x; idx < 16 * MT * (chunk / 8); idx += GEMM_WAVES * QIL_WAVE) {
      const int m = idx / (chunk / 8), c = (idx - m * (chunk / 8)) * 8;
      const uint4 v = c < width ? load_frag<ALIGNED>(A, m0 + m, M, kc + c, K) : make_uint4(0, 0, 0, 0);
      *reinterpret_cast<uint4*>(a_lds + m * row_width + c) = v;
    }
    __syncthreads();
    const int steps = (width + 31) / 32;
    for (int step = 0; step < steps; step += 2 * UNROLL) {
      request(b1, kc + (step + UNROLL) * 32);               // past k_end a request loads nothing
      multiply(b0, step, steps);
      request(b0, kc + (step + 2 * UNROLL) * 32);           // may be the first group of the next chunk
      multiply(b1, step + UNROLL, steps);
    }
  }
  // lane holds D[m = 4 kb + i][n = r] of each tile
  OUT* out = C + (size_t)split * M * N;
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int j = 0; j < NT; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = m0 + t * 16 + 4 * kb + i, n = n0 + j * 16 + r;
        if (m < M && n < N) store_out(out + (size_t)m * N + n, acc[t][j][i] + (bias ? bias[n] : 0.f));
      }
}

template <int MT, int NT, int UNROLL, typename OUT>
static int launch_stream(const bf16_t* A, const bf16_t* W, const float* bias, OUT* C, int M, int N, int K, int splits,
                         int chunk, hipStream_t s) {
  const int steps = (K + 31) / 32;
  const int steps_per_split = (steps + splits - 1) / splits;
  const int grain = 64 * UNROLL;                                         // the k loop runs in pairs of UNROLL steps
  if (chunk <= 0 || chunk > steps_per_split * 32) chunk = steps_per_split * 32;
  chunk = (chunk + grain - 1) / grain * grain;
  const size_t cap = 64 * 1024 / (16 * MT * sizeof(bf16_t));             // elements per row that fit 64 KB
  if ((size_t)chunk + GEMM_LDS_PAD > cap) chunk = (int)((cap - GEMM_LDS_PAD) / grain * grain);
  if (chunk < grain) return -1;
  const size_t lds = (size_t)16 * MT * (chunk + GEMM_LDS_PAD) * sizeof(bf16_t);
  dim3 grid((N + 128 * NT - 1) / (128 * NT), (M + 16 * MT - 1) / (16 * MT), splits);
  const bool aligned = (K % 8 == 0) && (((uintptr_t)A | (uintptr_t)W) % 16 == 0);
  if (aligned)
    hipLaunchKernelGGL((gemm_bf16_stream_kernel<MT, NT, UNROLL, true, OUT>), grid, dim3(GEMM_WAVES * QIL_WAVE), lds, s,
                       A, W, bias, C, M, N, K, steps_per_split, chunk);
  else
    hipLaunchKernelGGL((gemm_bf16_stream_kernel<MT, NT, UNROLL, false, OUT>), grid, dim3(GEMM_WAVES * QIL_WAVE), lds, s,
                       A, W, bias, C, M, N, K, steps_per_split, chunk);
  return 0;
}

// ---------------------------------------------------------------------------------------------------
// The same product with W read in whole cache lines.  The fragment layout above makes every load
// instruction touch 16 rows x 64 bytes; here a load instruction takes 4 rows x 256 contiguous bytes
// (lane l: row 4 u + l / 16, 16-byte piece l % 16), three stages of 16 rows x 128 columns are in
// flight in registers, and a stage passes through a wave-private 4 KB LDS buffer that turns it into
// fragments.  The 16-byte pieces of a row are stored at piece ^ row, so the writes (16 lanes, one
// row) and the fragment reads (16 lanes, 16 rows, one logical piece) both spread over all banks.
// LDS operations of one wave complete in program order, so the buffer needs no barrier.
// Takes M <= 16, K a multiple of 128 per split, 16-byte aligned operands, no bias.
#define LINES_WAVES 8

#define LINES_DEPTH 3                                      // stages of W in flight per wave
#define LINES_LDS_LIMIT (100 * 1024)                       // one block of 8 waves on a CU when A is long, two otherwise

// A given as the float32 residual stream whose RMSNorm is to be taken (qil/model.py:15-23), with the rows' sums of
// squares already there in pieces: squares [pieces][M], a piece for every 16 (or 8) columns of the stream, left by the kernel
// that completed the stream (gemm_bf16_add.hip).  The block adds the pieces in a fixed order, normalises its slice of the
// row (round, then the weight, as add_rmsnorm in elementwise.hip does) and needs no norm kernel before it.
struct NormedA {
  const float* stream;                                     // [M, K]
  const float* weight;                                     // [K]
  const float* squares;                                    // [pieces][M]
  int pieces;
  float eps;
};

// A block's slice of such an operand, columns k_begin .. k_begin + cols, on its way into LDS: ask() sends the first loads, put() waits for
// them (not for what was asked for in between) and leaves the rows in LDS, to be met behind a barrier.  M at most twice the waves.
// A wave adds the pieces of two rows' sums of squares; up to 512 of them (4,096 columns in pieces of 8, 8,192 in pieces of 16) are asked for
// together with what a thread's first two pieces of A are made of.  (Those past 256, asked for at their use, came back behind W: us
// a product, 12 rows of 6,144 x 2,560 in pieces of 8 11.3 -> 10.4, 1 and 16 of 7,168 x 5,120 in pieces of 16 15.4 -> 14.5 and 19.0 -> 18.1.)
// (All are held in place: the compiler otherwise moves loads whose use stands under a condition down to it.)
// MANY: more than 256 pieces (a choice at run time cost 0.1 us of 3.5 where they are fewer).
template <bool MANY>
struct NormedStage {
  static constexpr int EARLY = 2, SQUARES = 4;
  const NormedA& normed;
  float* rstd;                                             // 16 floats of LDS
  const int M, K, k_begin, pieces, all, threads, lane, wave, waves;
  float x[EARLY][8], g[EARLY][8], squares[2][SQUARES], more[2][SQUARES];
  __device__ __forceinline__ NormedStage(const NormedA& n, void* scratch, int m, int k, int first, int cols, int w, int ws)
      : normed(n), rstd(reinterpret_cast<float*>(scratch)), M(m), K(k), k_begin(first), pieces(cols / 8), all(m * (cols / 8)),
        threads(ws * QIL_WAVE), lane(threadIdx.x & (QIL_WAVE - 1)), wave(w), waves(ws) {}
  __device__ __forceinline__ void ask_piece(int idx, float (&to_x)[8], float (&to_g)[8]) {
    const int m = idx / pieces, c = (idx - m * pieces) * 8;
    ld8(normed.stream + (size_t)m * K + k_begin + c, to_x);
    ld8(normed.weight + k_begin + c, to_g);
  }
  __device__ __forceinline__ void ask_squares(int r2, int first, float (&to)[SQUARES]) {
#pragma unroll
    for (int i = 0; i < SQUARES; ++i)
      to[i] = normed.squares[(size_t)min(first + lane + i * QIL_WAVE, normed.pieces - 1) * M + min(wave + r2 * waves, M - 1)];
  }
  __device__ __forceinline__ void ask() {
#pragma unroll
    for (int r2 = 0; r2 < 2; ++r2)
      if (!r2 || M > waves) ask_squares(r2, 0, squares[r2]);
    if constexpr (MANY)
#pragma unroll
      for (int r2 = 0; r2 < 2; ++r2)
        if (!r2 || M > waves) ask_squares(r2, SQUARES * QIL_WAVE, more[r2]);
#pragma unroll
    for (int u = 0; u < EARLY; ++u)
      if (!u || all > threads) ask_piece(min((int)threadIdx.x + u * threads, all - 1), x[u], g[u]);
  }
  __device__ __forceinline__ void put_piece(int idx, const float (&from_x)[8], const float (&from_g)[8], bf16_t* a_lds, int row_width) {
    const int m = idx / pieces, c = (idx - m * pieces) * 8;
    const float scale = rstd[m];
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = round_to<bf16_t>(from_x[e] * scale) * from_g[e];
    *reinterpret_cast<uint4*>(a_lds + m * row_width + c) =
        make_uint4(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7]));
  }
  __device__ __forceinline__ void put(bf16_t* a_lds, int row_width) {
#pragma unroll
    for (int r2 = 0; r2 < 2; ++r2) {                        // (twice the waves: all rows there are)
      if (r2 && M <= waves) break;
      const int m = wave + r2 * waves;
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < SQUARES; ++i) {
        asm volatile("" : "+v"(squares[r2][i]));
        if (lane + i * QIL_WAVE < normed.pieces) sum += squares[r2][i];
      }
      if constexpr (MANY)
#pragma unroll
        for (int i = 0; i < SQUARES; ++i) {
          asm volatile("" : "+v"(more[r2][i]));
          if (lane + (SQUARES + i) * QIL_WAVE < normed.pieces) sum += more[r2][i];
        }
      for (int p = lane + (MANY ? 2 : 1) * SQUARES * QIL_WAVE; p < normed.pieces; p += QIL_WAVE) sum += normed.squares[(size_t)p * M + min(m, M - 1)];
      sum = wave_sum(sum);
      if (lane == 0 && m < M) rstd[m] = rsqrtf(sum / (float)K + normed.eps);
    }
#pragma unroll
    for (int u = 0; u < EARLY; ++u)
      if (!u || all > threads)
#pragma unroll
        for (int e = 0; e < 8; ++e) asm volatile("" : "+v"(x[u][e]), "+v"(g[u][e]));
    __syncthreads();
#pragma unroll
    for (int u = 0; u < EARLY; ++u)
      if ((int)threadIdx.x + u * threads < all) put_piece(threadIdx.x + u * threads, x[u], g[u], a_lds, row_width);
    for (int idx = threadIdx.x + EARLY * threads; idx < all; idx += threads) {
      ask_piece(idx, x[0], g[0]);
      put_piece(idx, x[0], g[0], a_lds, row_width);
    }
  }
};

// ASRC: 0 = A as it is, 1 = merged attention parts (UnmergedA), 2 = normalised stream (NormedA).  HOW, behind the merge (launch_lines):
// W's first requests go out ahead of the parts' arrival, or behind it, with a piece's loads all at once or its row's position first;
// behind the norm: NormedStage's MANY.
enum { AHEAD, AT_ONCE, POSITION_FIRST, MANY_SQUARES };
template <typename OUT, int ASRC, int WAVES = LINES_WAVES, int HOW = AHEAD>
__global__ void __launch_bounds__(WAVES * QIL_WAVE)
gemm_bf16_lines_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, OUT* __restrict__ C, int M, int N, int K,
                       int cols_per_split, UnmergedA unmerged, NormedA normed) {
  constexpr bool MERGE = ASRC == 1;
  extern __shared__ __align__(16) bf16_t lds[];            // A slice [8 or 16][cols + pad], then the waves' buffers
  const int lane = threadIdx.x & (QIL_WAVE - 1), wave = threadIdx.x / QIL_WAVE;
  const int r = lane & 15, kb = lane >> 4;
  const int a_rows = M <= 8 ? 8 : 16;                      // rows of A kept (8 or 16: a power of two)
  const int n0 = (blockIdx.x * WAVES + wave) * 16, split = blockIdx.z;
  const int k_begin = split * cols_per_split, stages = cols_per_split / 128;
  const int row_width = cols_per_split + GEMM_LDS_PAD;
  bf16_t* a_lds = lds;
  bf16_t* buffer = lds + a_rows * row_width + wave * (16 * 128);

  const int load_row = lane >> 4, piece = lane & 15;
  const bf16_t* source[4];                                 // rows past N read a valid row and are never stored
  int place[4];                                            // where this lane's piece of load u goes in the buffer
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int row = 4 * u + load_row;
    source[u] = W + (size_t)min(n0 + row, N - 1) * K + k_begin + piece * 8;
    place[u] = row * 128 + ((piece ^ row) & 15) * 8;
  }
  // Every wave walks its K range from a start of its own and wraps around: waves that all read the
  // same columns of their rows at the same time load a few memory channels only.
  const int turn = (n0 / 16) % stages;
  auto column = [&](int stage) { const int st = stage + turn; return (st >= stages ? st - stages : st) * 128; };
  // three stages in flight, each in registers of its own (named, so that none is indexed at run time)
  u32x4 w0[4], w1[4], w2[4];
  auto request = [&](u32x4 (&stage_w)[4], int stage) {
    const int at = column(stage);
#pragma unroll
    for (int u = 0; u < 4; ++u) stage_w[u] = load_once(source[u] + at);
  };
  auto request_first = [&]() {
    request(w0, 0);                                         // the host sees to stages >= 3
    request(w1, 1);
    request(w2, 2);
  };
  // What A is made of is asked for first and W's first stages right behind it, before anything is waited for (loads come back in
  // order, so waiting for A does not wait for W).  With W asked for behind A's arrival the two waits stood one behind the other: one
  // row of 4,096 x 1,024 behind the norm in 2 splits 5.1 -> 4.2 us, 8 rows 5.6 -> 5.1, 8 of 6,144 x 4,096 12.6 -> 12.2, 16 of 6,144 x 2,048
  // 9.0 -> 8.5 (a step of 28 layers and one row 966 -> 932 with the merge's part of it, launch_lines).
  constexpr int THREADS = WAVES * QIL_WAVE;
  const int pieces = cols_per_split / 8, all = M * pieces;  // (rows past M stay as they are in LDS: their products are never stored)
  if (ASRC == 2) {
    NormedStage<HOW == MANY_SQUARES> stage(normed, lds + a_rows * row_width + WAVES * (16 * 128), M, K, k_begin, cols_per_split, wave, WAVES);
    stage.ask();
    __builtin_amdgcn_sched_barrier(0);
    request_first();
    __builtin_amdgcn_sched_barrier(0);
    stage.put(a_lds, row_width);
  } else if (MERGE) {
    MergeParts<8, 4> parts;
    const int P = merge_part_keys(unmerged);
    int idx = threadIdx.x, m, c;
    auto ask = [&](int of) {
      m = of / pieces;
      c = (of - m * pieces) * 8;
      merge_ask(unmerged, P, m, k_begin + c, parts);
    };
    auto store = [&](const float (&v)[8]) {
      *reinterpret_cast<uint4*>(a_lds + m * row_width + c) =
          make_uint4(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7]));
    };
    auto put = [&]() {
      float v[8];
      merge_finish(unmerged, P, m, k_begin + c, parts, v);
      store(v);
    };
    if constexpr (HOW == AT_ONCE) {
      for (; idx < all; idx += THREADS) {
        ask(idx);
        put();
      }
      request_first();
    } else if constexpr (HOW == POSITION_FIRST) {
      for (; idx < all; idx += THREADS) {
        m = idx / pieces;
        c = (idx - m * pieces) * 8;
        float v[8];
        merged_values<8>(unmerged, m, k_begin + c, v);
        store(v);
      }
      request_first();
    } else if constexpr (WAVES < LINES_WAVES) {
      ask(min(idx, all - 1));
      __builtin_amdgcn_sched_barrier(0);
      request_first();
      parts.arrived();                                      // (in the loop this would be a wait for W as well)
      if (idx < all) put();
      for (idx += THREADS; idx < all; idx += THREADS) {
        ask(idx);
        put();
      }
    } else {
      ask(min(idx, all - 1));
      __builtin_amdgcn_sched_barrier(0);
      request(w0, 0);                                       // (all three stages of eight waves are in the way of the slower waves' parts)
      parts.arrived();
      if (idx < all) put();                                 // (a piece a thread: launch_lines)
      request(w1, 1);
      request(w2, 2);
    }
  } else {
    // A as it is goes from memory straight into LDS, 512 columns of a row an instruction, and is not waited for
    // here: W's first stages are asked for right behind it (loads complete in order, so waiting for A later
    // does not wait for them).  Rows past M repeat the last one; their products are never stored.
    const int row_loads = (cols_per_split + 511) / 512;
    for (int j = wave; j < a_rows * row_loads; j += WAVES) {
      const int m = __builtin_amdgcn_readfirstlane(j / row_loads), c0 = __builtin_amdgcn_readfirstlane(j - m * row_loads) * 512;
      if (c0 + lane * 8 < cols_per_split)
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) void*)(A + (size_t)min(m, M - 1) * K + k_begin + c0 + lane * 8),
            (__attribute__((address_space(3))) void*)(a_lds + m * row_width + c0), 16, 0, 0);
    }
    request_first();
  }
  if (ASRC == 0) {
    // A has landed, W's 12 loads need not: s_waitcnt vmcnt(12) lgkmcnt(0).  As a builtin and with the LDS counter
    // in it, because the compiler treats a load into LDS as an access of both kinds and, until it sees one wait
    // that covers both counters, makes every later wait for a load a wait for all of them.
    __builtin_amdgcn_s_waitcnt(0x07C);
    __builtin_amdgcn_s_barrier();
  } else {
    __syncthreads();
  }

  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  // lanes past the kept rows read the rows again: their products are rows of D that are never stored
  const bf16_t* a_row = a_lds + (r & (a_rows - 1)) * row_width + kb * 8;
  auto pass = [&](const u32x4 (&stage_w)[4]) {             // registers -> buffer
#pragma unroll
    for (int u = 0; u < 4; ++u) *reinterpret_cast<u32x4*>(buffer + place[u]) = stage_w[u];
  };
  auto multiply = [&](int stage) {
    const int at = column(stage);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      const u32x4 b = *reinterpret_cast<const u32x4*>(buffer + r * 128 + (((4 * s4 + kb) ^ r) & 15) * 8);
      const u32x4 a = *reinterpret_cast<const u32x4*>(a_row + at + s4 * 32);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0,
                                                    0, 0);
    }
    __builtin_amdgcn_wave_barrier();
  };
  int stage = 0;
  for (; stage + 6 <= stages; stage += 3) {                 // every stage here has a successor three ahead
    pass(w0); request(w0, stage + 3); multiply(stage);
    pass(w1); request(w1, stage + 4); multiply(stage + 1);
    pass(w2); request(w2, stage + 5); multiply(stage + 2);
  }
  // the last three to five stages: requests run out
  const int left = stages - stage;
  pass(w0); if (left > 3) request(w0, stage + 3); multiply(stage);
  pass(w1); if (left > 4) request(w1, stage + 4); multiply(stage + 1);
  pass(w2); multiply(stage + 2);
  if (left > 3) { pass(w0); multiply(stage + 3); }
  if (left > 4) { pass(w1); multiply(stage + 4); }
  OUT* out = C + (size_t)split * M * N;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = 4 * kb + i, n = n0 + r;
    if (m < M && n < N) store_out(out + (size_t)m * N + n, acc[i]);
  }
}

static size_t lines_lds(int M, int K, int splits, int waves = LINES_WAVES) {
  const int rows = M <= 8 ? 8 : 16;
  return ((size_t)rows * (K / splits + GEMM_LDS_PAD) + (size_t)waves * 16 * 128) * sizeof(bf16_t) + 16 * sizeof(float);
}

// Whether the whole-line kernel takes the product with this many splits.
static bool lines_takes(const void* A, const void* W, const float* bias, int M, int N, int K, int splits) {
  if (bias || M > 16 || N < 1 || K % (128 * splits) || K / (128 * splits) < LINES_DEPTH ||
      (((uintptr_t)A | (uintptr_t)W) % 16))
    return false;
  return lines_lds(M, K, splits) <= LINES_LDS_LIMIT;
}

template <typename OUT, int ASRC, int WAVES, int HOW = AHEAD>
static int launch_lines_waves(const bf16_t* A, const bf16_t* W, OUT* C, int M, int N, int K, int splits, hipStream_t s,
                              UnmergedA unmerged, NormedA normed) {
  const size_t lds = lines_lds(M, K, splits, WAVES);
  auto kernel = gemm_bf16_lines_kernel<OUT, ASRC, WAVES, HOW>;
  static size_t granted = 0;                              // per instantiation
  if (lds > 64 * 1024 && lds > granted) {
    hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
    granted = lds;
  }
  dim3 grid((N + 16 * WAVES - 1) / (16 * WAVES), 1, splits);
  hipLaunchKernelGGL(kernel, grid, dim3(WAVES * QIL_WAVE), lds, s, A, W, C, M, N, K, K / splits, unmerged, normed);
  return 0;
}

// Blocks of 4 waves where those of 8 leave half of the CUs without one: a CU draws 36 GB/s at most.  One row, inside a step:
// 1,024 x 2,048 behind the merge in 4 splits 6.0 us with 32 blocks of 8, 4.6 with 64 of 4; 4,096 x 1,024 behind the norm in 2 5.9 with
// 64, 5.4 with 128 (its operands asked for in one batch); 8 rows of 2,048 x 2,048 in 4 5.3 with 64, 4.5 with 128.  Up to 8 rows:
// with 16 half the threads stage twice the rows.  Behind the merge up to 4 rows: every block merges all of its rows' parts, and twice
// the blocks of half the threads take longer for that than they gain (8 rows and 63 parts 16.7 us with 8 waves, 22.5 with 4; 6 rows
// and 2 parts 5.5 / 5.9; 4 rows 4 is ahead at any number of parts).
// Behind the merge W's first stages are asked for ahead of the parts' arrival (AHEAD) where all parts come in one turn: up to four of
// them for blocks of 4 waves, a piece of A a thread for those of 8; a second turn's loads would come back behind W, which pays only where
// a quarter of the threads have none and W is much.  us without / with: 1 row of 1,024 x 2,048, 2 parts 4.5 / 4.4 alone and 5.7 / 5.3 inside a
// step, 9 parts 5.9 / 5.9; 8 rows of 4,096 x 4,096, 4 parts 8.7 / 8.1, 8 level, 6 rows and 8 parts 10.3 / 9.6, of 1,024 x 2,048 6.9 / 7.5; 16
// rows of 1,024 x 2,048, 2 parts (two pieces a thread) 6.8 / 7.2.
// Where they are not, blocks of 8 waves with up to two pieces a thread ask for the row's position first, others for all of a piece at
// once (us position first / at once: 16 rows of 1,024 x 2,048, 2 parts 6.8 / 7.2, 8 of 896 x 896 8.3 / 8.7, but 16 of 896 x 896 (3.5 pieces) 10.2 / 9.8,
// 12 of 5,120 x 8,192 24.3 / 23.7, and 2 of 1,024 x 2,048, 16 parts in blocks of 4 waves 6.5 / 6.2).
#define LINES_FEW_WAVES 4
template <typename OUT, int ASRC = 0>
static int launch_lines(const bf16_t* A, const bf16_t* W, OUT* C, int M, int N, int K, int splits, hipStream_t s,
                        UnmergedA unmerged = UnmergedA(), NormedA normed = NormedA()) {
  const long blocks = (long)((N + 16 * LINES_WAVES - 1) / (16 * LINES_WAVES)) * splits;
  const bool few = M <= (ASRC == 1 ? 4 : 8) && blocks <= QIL_CUS / 2;
  if constexpr (ASRC == 1) {
    constexpr int THREADS = LINES_WAVES * QIL_WAVE;
    const long pieces = (long)M * (K / splits / 8);
    if (few && unmerged.parts > 4) return launch_lines_waves<OUT, ASRC, LINES_FEW_WAVES, AT_ONCE>(A, W, C, M, N, K, splits, s, unmerged, normed);
    if (!few && pieces > 2 * THREADS) return launch_lines_waves<OUT, ASRC, LINES_WAVES, AT_ONCE>(A, W, C, M, N, K, splits, s, unmerged, normed);
    if (!few && pieces > (unmerged.parts <= 4 ? THREADS : blocks > QIL_CUS / 2 ? THREADS * 3 / 4 : 0))
      return launch_lines_waves<OUT, ASRC, LINES_WAVES, POSITION_FIRST>(A, W, C, M, N, K, splits, s, unmerged, normed);
  }
  if constexpr (ASRC == 2)
    if (normed.pieces > 256)
      return few ? launch_lines_waves<OUT, ASRC, LINES_FEW_WAVES, MANY_SQUARES>(A, W, C, M, N, K, splits, s, unmerged, normed)
                 : launch_lines_waves<OUT, ASRC, LINES_WAVES, MANY_SQUARES>(A, W, C, M, N, K, splits, s, unmerged, normed);
  if (few) return launch_lines_waves<OUT, ASRC, LINES_FEW_WAVES>(A, W, C, M, N, K, splits, s, unmerged, normed);
  return launch_lines_waves<OUT, ASRC, LINES_WAVES>(A, W, C, M, N, K, splits, s, unmerged, normed);
}

// ---------------------------------------------------------------------------------------------------
// The whole-line product for 17 to 192 rows of A and any length of K.  A does not stay in LDS as a whole
// slice: it passes through it one stage (128 columns) at a time, in two slots that the block's threads
// fill in turn, from registers that are loaded three stages ahead, as W's are.  One barrier a stage: the
// stage's slot has been written before it and the other slot may be written after it.  All waves of a
// block are at the same stage, so the walk through K starts at a column of the block's (not the wave's) own.
// MT: 16-row tiles of A (M <= 16 MT); every W fragment read from the buffer serves MT products.
// Takes 8 < M <= 192, K a multiple of 128 per split with at least 3 stages, 16-byte aligned operands, no bias.
#define CHUNK_ROW (128 + GEMM_LDS_PAD)
#define CHUNKS_MOST_ROWS 192

// GATED: W is the [N = 2 inner, K] matrix of a gated feed-forward with gate and up rows interleaved in tiles of 16
// (gate rows 0-15, up rows 0-15, gate rows 16-31, ...), and C [M, inner] gets act(A gate^T, A up^T)
// (gated_act.h; qil/model.py:71).  A block then owns 64 columns of `inner`, 128 consecutive rows of W: the even waves make gate
// products, the odd waves the up products that belong to them; these hand their sums over in LDS and the even waves
// store the activations.  K is not split: no partial sums in memory and no separate activation pass.  (With the gate
// rows stacked before the up rows a block would read two regions a power of two apart at the same columns at the
// same time, which loads a few memory channels only: 59 us against 45 for 64 rows at 8B sizes.)
template <typename OUT, int MT, int GATED = QIL_UNGATED>
__global__ void __launch_bounds__(LINES_WAVES * QIL_WAVE)
gemm_bf16_chunks_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, OUT* __restrict__ C, int M, int N,
                        int K, int cols_per_split, GateFn fn) {
  extern __shared__ __align__(16) bf16_t lds[];            // two stages of A [16 MT][128 + pad], then the waves' buffers
  constexpr int A_ROWS = 16 * MT, SLOT = A_ROWS * CHUNK_ROW;
  constexpr int PIECES = A_ROWS * 16 / (LINES_WAVES * QIL_WAVE);   // 16-byte pieces of a stage of A per thread
  static_assert(PIECES >= 1, "a stage of A has fewer pieces than the block has threads");
  const int lane = threadIdx.x & (QIL_WAVE - 1), wave = threadIdx.x / QIL_WAVE;
  const int r = lane & 15, kb = lane >> 4;
  const int split = blockIdx.z;
  const int inner_n0 = (blockIdx.x * (LINES_WAVES / 2) + (wave >> 1)) * 16;  // GATED: the wave's column of the result
  const int n0 = (blockIdx.x * LINES_WAVES + wave) * 16;
  const int k_begin = split * cols_per_split, stages = cols_per_split / 128;
  bf16_t* buffer = lds + 2 * SLOT + wave * (16 * 128);

  const int load_row = lane >> 4, piece = lane & 15;
  const bf16_t* source[4];                                 // rows past N read a valid row and are never stored
  int place[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int row = 4 * u + load_row;
    source[u] = W + (size_t)min(n0 + row, N - 1) * K + k_begin + piece * 8;
    place[u] = row * 128 + ((piece ^ row) & 15) * 8;
  }
  // This thread's pieces of a stage of A.  Rows past M read row M - 1: their products land in rows of the
  // result that are never stored.  (A load under a condition would make the compiler wait for every load in
  // flight, W's too, at each stage.)
  const bf16_t* a_source[PIECES];
  int a_place[PIECES];
#pragma unroll
  for (int u = 0; u < PIECES; ++u) {
    const int p = threadIdx.x + u * (LINES_WAVES * QIL_WAVE), row = p >> 4, pc = p & 15;
    a_source[u] = A + (size_t)min(row, M - 1) * K + k_begin + pc * 8;
    a_place[u] = row * CHUNK_ROW + pc * 8;
  }
  const int turn = blockIdx.x % stages;
  auto column = [&](int stage) { const int st = stage + turn; return (st >= stages ? st - stages : st) * 128; };
  u32x4 w0[4], w1[4], w2[4], a0[PIECES], a1[PIECES], a2[PIECES];
  auto request = [&](u32x4 (&stage_w)[4], int stage) {
    const int at = column(stage);
#pragma unroll
    for (int u = 0; u < 4; ++u) stage_w[u] = load_once(source[u] + at);
  };
  auto request_a = [&](u32x4 (&stage_a)[PIECES], int stage) {
    const int at = column(stage);
#pragma unroll
    for (int u = 0; u < PIECES; ++u) stage_a[u] = *reinterpret_cast<const u32x4*>(a_source[u] + at);
  };
  auto store_a = [&](const u32x4 (&stage_a)[PIECES], int stage) {
    bf16_t* slot = lds + (stage & 1) * SLOT;
#pragma unroll
    for (int u = 0; u < PIECES; ++u) *reinterpret_cast<u32x4*>(slot + a_place[u]) = stage_a[u];
  };
  request_a(a0, 0); request_a(a1, 1); request_a(a2, 2);     // the host sees to stages >= 3
  request(w0, 0); request(w1, 1); request(w2, 2);
  store_a(a0, 0);
  if (3 < stages) request_a(a0, 3);
  __syncthreads();

  f32x4 acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  auto pass = [&](const u32x4 (&stage_w)[4]) {             // registers -> buffer
#pragma unroll
    for (int u = 0; u < 4; ++u) *reinterpret_cast<u32x4*>(buffer + place[u]) = stage_w[u];
  };
  auto multiply = [&](int stage) {
    const bf16_t* a_row = lds + (stage & 1) * SLOT + r * CHUNK_ROW + kb * 8;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      const u32x4 b = *reinterpret_cast<const u32x4*>(buffer + r * 128 + (((4 * s4 + kb) ^ r) & 15) * 8);
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const u32x4 a = *reinterpret_cast<const u32x4*>(a_row + t * 16 * CHUNK_ROW + s4 * 32);
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b),
                                                         acc[t], 0, 0, 0);
      }
    }
    __builtin_amdgcn_wave_barrier();
  };
  // Stage s: its W goes from registers w to the buffer; registers a hold stage s + 1 of A.  `inner`: every
  // request of the stage has a target.  (A request under a condition, even a uniform one, makes the compiler
  // wait for all loads in flight at the next use of any of them, so the stages that need conditions are apart.)
  auto step = [&](int s, u32x4 (&w)[4], u32x4 (&a)[PIECES], auto inner) {
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
  if (GATED) {
    // every step ends with a barrier: the slots of A are free.  [up wave][tile][lane][4] floats
    float* handed = reinterpret_cast<float*>(lds);
    if (wave & 1)
#pragma unroll
      for (int t = 0; t < MT; ++t) *reinterpret_cast<f32x4*>(handed + (((wave >> 1) * MT + t) * QIL_WAVE + lane) * 4) = acc[t];
    __syncthreads();
    if (!(wave & 1)) {
      const int inner = N / 2;
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const f32x4 up = *reinterpret_cast<const f32x4*>(handed + (((wave >> 1) * MT + t) * QIL_WAVE + lane) * 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int m = t * 16 + 4 * kb + i, n = inner_n0 + r;
          const float g = acc[t][i];
          if (m < M && n < inner) store_out(C + (size_t)m * inner + n, gate_by<GATED == QIL_GATED_SILU>(g, up[i], fn));
        }
      }
    }
    return;
  }
  OUT* out = C + (size_t)split * M * N;
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = t * 16 + 4 * kb + i, n = n0 + r;
      if (m < M && n < N) store_out(out + (size_t)m * N + n, acc[t][i]);
    }
}

// (9 to 16 rows come here when the whole-line kernel cannot keep their slice of A in LDS: 16 rows of 4,096 columns and
// the waves' buffers are 64 bytes more than a CU has; the logits of such a step took 275 us on the fragment-layout
// kernel.)
static bool chunks_takes(const void* A, const void* W, const float* bias, int M, int N, int K, int splits) {
  return !bias && M > 8 && M <= CHUNKS_MOST_ROWS && N >= 1 && splits >= 1 && K % (128 * splits) == 0 &&
         K / (128 * splits) >= LINES_DEPTH && (((uintptr_t)A | (uintptr_t)W) % 16) == 0;
}

// K splits of that kernel when partial sums are allowed: the most (a power of two up to 8, with at least
// three stages each) that keep the blocks within the 256 CUs; one block a CU runs them all at once, and of the
// numbers of splits tried (1 to 8 for the products of 8B and 32B layer sizes) this one was the fastest each time.
static int chunks_splits(int N, int K) {
  const long tiles = (N + 16 * LINES_WAVES - 1) / (16 * LINES_WAVES);
  int splits = 1;
  for (int c = 2; c <= 8; c *= 2)
    if (tiles * c <= QIL_CUS && K % (128 * c) == 0 && K / (128 * c) >= LINES_DEPTH) splits = c;
  return splits;
}

template <typename OUT, int MT, int GATED = false>
static int launch_chunks_tiles(const bf16_t* A, const bf16_t* W, OUT* C, int M, int N, int K, int splits, GateFn fn, hipStream_t s) {
  const size_t lds = ((size_t)2 * 16 * MT * CHUNK_ROW + (size_t)LINES_WAVES * 16 * 128) * sizeof(bf16_t);
  auto kernel = gemm_bf16_chunks_kernel<OUT, MT, GATED>;
  static size_t granted = 0;                              // per instantiation
  if (lds > 64 * 1024 && lds > granted) {
    hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
    granted = lds;
  }
  // GATED: a block owns 64 columns of the result (N / 2 of them), else 128 of N
  dim3 grid(GATED ? (N / 2 + 63) / 64 : (N + 16 * LINES_WAVES - 1) / (16 * LINES_WAVES), 1, splits);
  hipLaunchKernelGGL(kernel, grid, dim3(LINES_WAVES * QIL_WAVE), lds, s, A, W, C, M, N, K, K / splits, fn);
  return 0;
}

template <typename OUT, int GATED = QIL_UNGATED>
static int launch_chunks(const bf16_t* A, const bf16_t* W, OUT* C, int M, int N, int K, int splits, hipStream_t s, GateFn fn = {}) {
  if (M <= 32) return launch_chunks_tiles<OUT, 2, GATED>(A, W, C, M, N, K, splits, fn, s);
  if (M <= 64) return launch_chunks_tiles<OUT, 4, GATED>(A, W, C, M, N, K, splits, fn, s);
  if (M <= 96) return launch_chunks_tiles<OUT, 6, GATED>(A, W, C, M, N, K, splits, fn, s);
  if (M <= 128) return launch_chunks_tiles<OUT, 8, GATED>(A, W, C, M, N, K, splits, fn, s);
  if (M <= 160) return launch_chunks_tiles<OUT, 10, GATED>(A, W, C, M, N, K, splits, fn, s);
  return launch_chunks_tiles<OUT, 12, GATED>(A, W, C, M, N, K, splits, fn, s);
}

// ---------------------------------------------------------------------------------------------------
// Gate and up products of a gated feed-forward with the activation in the epilogue:
//   out[m, n] = act(A W[n]^T, A W[inner + n]^T),  n < inner        (gated_act.h; qil/model.py:71)
// W is the [2 inner, K] matrix with the gate rows stacked before the up rows, or with both interleaved in tiles of
// 16 rows (gate rows 0-15, up rows 0-15, gate rows 16-31, ...).  A "pair" is 16 gate rows and the 16 up rows
// that belong to them.  A block owns `pairs` consecutive pairs and `ksplit` waves per pair, which split
// K among themselves and add their float32 sums in LDS in wave order, so nothing but the finished
// activations leaves the block: no partial sums in memory and no separate activation pass.  All of A
// (8 or 16 rows) sits in LDS once per block.  W is read in whole cache lines as in the kernel above
// (two stages in flight, gate and up taking turns in the wave's buffer).
// Takes M <= 16 (while A fits in LDS), inner a multiple of 16, K a multiple of 128 ksplit with at least 2 stages a wave,
// 16-byte aligned operands.
#define GATED_MAX_WAVES 12                                 // three waves a SIMD: 168 registers each
#define GATED_ROWS_FEWEST_BLOCKS 128                       // of the 17-to-192-row kernel: see gated_rows_takes
#define GATED_ROWS_MOST 64                                 // beyond, the product and a separate activation are faster

// NORMED: A is the norm of the residual stream (NormedA), made by every block while W is on its way (M at most twice the waves).
template <typename OUT, bool SILU, bool NORMED = false>
__global__ void __launch_bounds__(GATED_MAX_WAVES * QIL_WAVE)
gemm_bf16_gated_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, OUT* __restrict__ out, int M,
                       int inner, int K, int ksplit, int interleaved, GateFn fn, NormedA normed) {
  extern __shared__ __align__(16) bf16_t lds[];            // A [8 or 16][K + pad], then a 4 KB buffer per wave
  const int a_rows = M <= 8 ? 8 : 16;                      // rows of A kept (8 or 16: a power of two)
  const int lane = threadIdx.x & (QIL_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / QIL_WAVE);
  const int r = lane & 15, kb = lane >> 4;
  const int pair = wave / ksplit, part = wave - pair * ksplit;
  const int pairs = blockDim.x / QIL_WAVE / ksplit;
  // a pair past the end repeats the last one and stores nothing
  const int n0 = min(blockIdx.x * pairs + pair, inner / 16 - 1) * 16;
  const bool stores = (blockIdx.x * pairs + pair) * 16 < inner;
  const int cols_per_wave = K / ksplit, k_begin = part * cols_per_wave, stages = cols_per_wave / 128;
  const int row_width = K + GEMM_LDS_PAD;
  bf16_t* a_lds = lds;
  bf16_t* buffer = lds + a_rows * row_width + wave * (16 * 128);

  // this lane's part of a stage: rows 4 u + lane / 16 (u < 4), 16-byte piece lane % 16, stored at piece ^ row
  const int load_row = lane >> 4, piece = lane & 15;
  const bf16_t* gate_source[4];
  int place[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int row = 4 * u + load_row;
    gate_source[u] = W + (size_t)((interleaved ? 2 * n0 : n0) + row) * K + k_begin + piece * 8;
    place[u] = row * 128 + ((piece ^ row) & 15) * 8;
  }
  // the up rows of a pair: `inner` rows after its gate rows (stacked), or right after them (interleaved in tiles of 16)
  const size_t up_offset = (size_t)(interleaved ? 16 : inner) * K;
  // Every wave walks its K range from a start of its own and wraps around: waves that all read the
  // same columns of their rows at the same time load a few memory channels only.
  const int turn = (n0 / 16) % stages;
  auto column = [&](int stage) { const int st = stage + turn; return (st >= stages ? st - stages : st) * 128; };

  u32x4 g0[4], u0[4], g1[4], u1[4];                        // two stages, named so that none is indexed at run time
  auto request = [&](u32x4 (&w)[4], size_t offset, int stage) {
    const int at = column(stage);
#pragma unroll
    for (int u = 0; u < 4; ++u) w[u] = load_once(gate_source[u] + offset + at);
  };
  // A goes straight into LDS, 512 columns of a row an instruction, with W's first two stages asked for right behind it: loads complete
  // in order, so A is waited for without W, and W without A.  (In registers, with A behind W, A was there when all of W's first
  // requests were, and with A ahead W was asked for only when A was there: 3,072 x 1,024,
  // one row 5.3 -> 4.6 us, 16 rows 6.4 -> 5.3; 9,728 x 2,560, 8 rows 19.9 -> 19.2, 16 rows 20.5 -> 19.4.)  Rows past M stay as they are in LDS: their products are rows of D that are never stored.
  const int waves = blockDim.x / QIL_WAVE;
  auto request_first = [&]() {
    request(g0, 0, 0); request(u0, up_offset, 0);           // the host sees to stages >= 2
    request(g1, 0, 1); request(u1, up_offset, 1);
  };
  if constexpr (NORMED) {
    NormedStage<false> stage(normed, lds + a_rows * row_width + waves * (16 * 128), M, K, 0, K, wave, waves);
    stage.ask();
    __builtin_amdgcn_sched_barrier(0);
    request_first();
    __builtin_amdgcn_sched_barrier(0);
    stage.put(a_lds, row_width);
    __syncthreads();
  } else {
    for (int c0 = 0; c0 < K; c0 += 512)
      if (c0 + lane * 8 < K) {
        const bf16_t* from = A + (size_t)wave * K + c0 + lane * 8;
        bf16_t* to = a_lds + wave * row_width + c0;
#pragma unroll 4
        for (int m = wave; m < M; m += waves) {
          __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)from,
                                           (__attribute__((address_space(3))) void*)to, 16, 0, 0);
          from += (size_t)waves * K;
          to += waves * row_width;
        }
      }
    request_first();
    __builtin_amdgcn_s_waitcnt(0x4070);                     // vmcnt(16) lgkmcnt(0): see the whole-line kernel
    __builtin_amdgcn_s_barrier();
  }

  f32x4 gate = {0.f, 0.f, 0.f, 0.f}, up = {0.f, 0.f, 0.f, 0.f};
  // lanes past the kept rows read the rows again: their products are rows of D that are never stored
  const bf16_t* a_row = a_lds + (r & (a_rows - 1)) * row_width + k_begin + kb * 8;
  auto pass = [&](const u32x4 (&w)[4]) {                   // registers -> buffer
#pragma unroll
    for (int u = 0; u < 4; ++u) *reinterpret_cast<u32x4*>(buffer + place[u]) = w[u];
  };
  auto multiply = [&](int stage, f32x4& acc) {
    const int at = column(stage);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      const u32x4 b = *reinterpret_cast<const u32x4*>(buffer + r * 128 + (((4 * s4 + kb) ^ r) & 15) * 8);
      const u32x4 a = *reinterpret_cast<const u32x4*>(a_row + at + s4 * 32);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0,
                                                    0, 0);
    }
    __builtin_amdgcn_wave_barrier();
  };
  int stage = 0;
  for (; stage + 4 <= stages; stage += 2) {                 // both stages here have a successor two ahead
    pass(g0); request(g0, 0, stage + 2); multiply(stage, gate);
    pass(u0); request(u0, up_offset, stage + 2); multiply(stage, up);
    pass(g1); request(g1, 0, stage + 3); multiply(stage + 1, gate);
    pass(u1); request(u1, up_offset, stage + 3); multiply(stage + 1, up);
  }
  const bool three = stages - stage == 3;                   // two or three stages are left
  pass(g0); if (three) request(g0, 0, stage + 2);
  multiply(stage, gate);
  pass(u0); if (three) request(u0, up_offset, stage + 2);
  multiply(stage, up);
  pass(g1); multiply(stage + 1, gate);
  pass(u1); multiply(stage + 1, up);
  if (three) {
    pass(g0); multiply(stage + 2, gate);
    pass(u0); multiply(stage + 2, up);
  }

  // the waves' sums meet in LDS (each wave's in its own buffer, which it has finished with): [gate, up][lane][4]
  float* sums = reinterpret_cast<float*>(lds + a_rows * row_width);
  constexpr int BUFFER = 16 * 128 / 2;                       // floats of a wave's buffer
  *reinterpret_cast<f32x4*>(sums + wave * BUFFER + lane * 4) = gate;
  *reinterpret_cast<f32x4*>(sums + wave * BUFFER + (QIL_WAVE + lane) * 4) = up;
  __syncthreads();
  if (part == 0 && stores) {
    f32x4 g = {0.f, 0.f, 0.f, 0.f}, v = {0.f, 0.f, 0.f, 0.f};
    for (int w = wave; w < wave + ksplit; ++w) {            // fixed order
      g += *reinterpret_cast<const f32x4*>(sums + w * BUFFER + lane * 4);
      v += *reinterpret_cast<const f32x4*>(sums + w * BUFFER + (QIL_WAVE + lane) * 4);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = 4 * kb + i, n = n0 + r;                 // lane holds D[m = 4 kb + i][n = r]
      if (m < M) store_out(out + (size_t)m * inner + n, gate_by<SILU>(g[i], v[i], fn));
    }
  }
}

// The block shape of the gated kernel for these sizes (pairs a block, waves a pair); false if it does
// not take them.
static size_t gated_lds(int M, int K, int waves) {
  return ((size_t)(M <= 8 ? 8 : 16) * (K + GEMM_LDS_PAD) + (size_t)waves * 16 * 128) * sizeof(bf16_t);
}

static bool gated_plan(const void* A, const void* W, int M, int inner, int K, int* pairs, int* ksplit) {
  if (M < 1 || M > 16 || inner < 16 || inner % 16 || K % 128 || (((uintptr_t)A | (uintptr_t)W) % 16))
    return false;
  // Most waves a pair that still leave 16 stages each; while the waves of all pairs are fewer than the machine
  // holds (256 CUs x 8), 2 stages each will do: a small product is bound by the loads in flight, not by LDS sums.
  int ks = 0;
  for (int c = 8; c >= 1 && !ks; c /= 2)
    if (K % (128 * c) == 0 && K / (128 * c) >= (c == 1 || (long)(inner / 16) * c <= 8 * QIL_CUS ? 2 : 16)) ks = c;
  if (!ks) return false;
  // Pairs that are fewer than the CUs: a CU each, and up to four waves with two stages or more, all on their way at once where they
  // are two (8 rows, two waves / four: 3,072 x 1,024 5.3 / 5.3 us, 4,096 x 4,096 13.9 / 13.3, with eight 16.4; one / two: 768 x 512
  // 4.3 / 3.7, 2,048 x 768 5.6 / 4.9).
  if (inner / 16 <= QIL_CUS && gated_lds(M, K, 8) <= 156 * 1024) {
    *pairs = 1;
    *ksplit = 1;
    for (int c = 2; c <= 4; c *= 2)
      if (K % (128 * c) == 0 && K / (128 * c) >= 2) *ksplit = c;
    return true;
  }
  // Pairs a block: what a CU has to do in all (its blocks one after the other, as many at a time as LDS and
  // the 12 wave slots allow) over how well its waves keep memory busy (8 or more do).  Ties go to more pairs.
  const int all_pairs = inner / 16;
  int best = 0;
  double best_cost = 0;
  for (int pb = GATED_MAX_WAVES / ks; pb >= 1; --pb) {
    const size_t lds = gated_lds(M, K, pb * ks);
    if (lds > 156 * 1024) continue;
    const long resident = std::max<long>(1, std::min<long>((160 * 1024) / lds, GATED_MAX_WAVES / (pb * ks)));
    const long blocks = (all_pairs + pb - 1) / pb, per_cu = (blocks + QIL_CUS - 1) / QIL_CUS;
    const long together = std::min(resident, per_cu), rounds = (per_cu + together - 1) / together;
    const double cost = (double)rounds * pb * 8.0 / (double)std::min<long>(8, together * pb * ks);
    if (!best || cost < best_cost) { best = pb; best_cost = cost; }
  }
  if (!best) return false;
  *pairs = best;
  *ksplit = ks;
  // A large product is bound by memory, and what counts is how its blocks fall on the CUs.  Measured with the weights
  // read once (nontemporal loads): a CU draws at most 36 GB/s, and 7.3 GB/s for every wave it holds (two stages of a
  // gate and an up tile in flight each), the chip 6.8 TB/s; blocks run in rounds of one (or, where LDS and wave slots
  // allow, two) a CU, a round costs 2 us beside its bytes, and a block 4 ns for its copy of A.  Of all shapes that
  // fit, the one with the least time by this count: at 32B sizes 7 pairs of one wave each (229 blocks, one round:
  // 80 us) instead of 4 pairs of two waves (400 blocks: 87 us); at 8B sizes the choice above.
  const double bytes = 2.0 * inner * (double)K * sizeof(bf16_t);
  if (bytes >= 96e6) {
    double least = 0;
    for (int c = 1; c <= 8; c *= 2) {
      if (K % (128 * c) || K / (128 * c) < 2) continue;
      for (int pb = 1; pb * c <= GATED_MAX_WAVES; ++pb) {
        const size_t lds = gated_lds(M, K, pb * c);
        if (lds > 156 * 1024) continue;
        const long resident = std::max<long>(1, std::min<long>((160 * 1024) / lds, GATED_MAX_WAVES / (pb * c)));
        const long blocks = (all_pairs + pb - 1) / pb, round = QIL_CUS * resident;
        const double block_bytes = bytes * pb / all_pairs;
        double time = 0.004 * blocks;
        for (long left = blocks; left > 0; left -= round) {
          const long now = std::min(left, round), cus = std::min<long>(QIL_CUS, now);
          const double waves_a_cu = (double)now / cus * pb * c;
          const double rate = std::min(6800.0, cus * std::min(36.0, 7.3 * waves_a_cu));   // GB/s
          time += now * block_bytes / (rate * 1e3) + 2.0;                                 // us
        }
        if (least == 0 || time < least) { least = time; *pairs = pb; *ksplit = c; }
      }
    }
  }
  return true;
}

// 17 to 64 rows of a matrix with interleaved rows: the kernel that passes A through LDS in stages, with the gate's
// epilogue.  It cannot split K, so it needs enough blocks of 64 result columns to fill the chip (`fewest`: 0 = the
// measured bound, tests pass 1).  Measured against the product followed by the activation kernel, 64 rows: 45.0
// against 47.6 us at 8B sizes (192 blocks), 108 against 117 at 32B sizes (400), 29 against 31 at 4B sizes (152); with
// 128 rows the fused kernel loses (74 against 55 at 8B sizes: its 8 row tiles leave a wave too few registers).
static bool gated_rows_takes(const void* A, const void* W, int M, int inner, int K, int interleaved, int fewest) {
  if (!interleaved || M <= 16 || M > GATED_ROWS_MOST || inner < 16 || inner % 16 || K % 128 || K / 128 < LINES_DEPTH ||
      (((uintptr_t)A | (uintptr_t)W) % 16))
    return false;
  return (inner + 63) / 64 >= (fewest ? fewest : GATED_ROWS_FEWEST_BLOCKS);
}

extern "C" int qil_gemm_bf16_gated_takes(int M, int inner, int K, int interleaved) {
  int pairs, ksplit;
  return gated_plan(nullptr, nullptr, M, inner, K, &pairs, &ksplit) ||
         gated_rows_takes(nullptr, nullptr, M, inner, K, interleaved, 0);
}

// out [M, inner] of out_dtype = act(A W[:inner]^T, A W[inner:]^T), act, limit, alpha: a gate function of gated_act.h.
// pairs, ksplit: 0 = chosen here (tuning runs set them).
extern "C" int qil_gemm_bf16_gated_act(const void* A, const void* W, void* out, int M, int inner, int K, int out_dtype,
                                       int pairs, int ksplit, int interleaved, int act, float limit, float alpha,
                                       hipStream_t s) {
  if (!gate_fn_known(act)) return -1;
  const GateFn fn{act, limit, alpha};
  if (M == 0 || inner == 0) return 0;
  if (M > 16) {                                              // pairs: the fewest blocks to accept (tests pass 1)
    if (!gated_rows_takes(A, W, M, inner, K, interleaved, pairs)) return -1;
#define QIL_CHUNKS_GATED(OUT, GATED) \
  launch_chunks<OUT, GATED>((const bf16_t*)A, (const bf16_t*)W, (OUT*)out, M, 2 * inner, K, 1, s, fn)
    const int status = out_dtype == QIL_F32 ? (act == QIL_ACT_SILU ? QIL_CHUNKS_GATED(float, QIL_GATED_SILU) : QIL_CHUNKS_GATED(float, QIL_GATED_OTHER))
                                            : (act == QIL_ACT_SILU ? QIL_CHUNKS_GATED(bf16_t, QIL_GATED_SILU) : QIL_CHUNKS_GATED(bf16_t, QIL_GATED_OTHER));
#undef QIL_CHUNKS_GATED
    if (status) return status;
    QIL_RETURN_LAUNCH_STATUS();
  }
  int planned_pairs, planned_ksplit;
  if (!gated_plan(A, W, M, inner, K, &planned_pairs, &planned_ksplit)) return -1;
  if (!pairs) pairs = planned_pairs;
  if (!ksplit) ksplit = planned_ksplit;
  if (pairs < 1 || ksplit < 1 || pairs * ksplit > GATED_MAX_WAVES || K % (128 * ksplit) || K / (128 * ksplit) < 2) return -1;
  const size_t lds = gated_lds(M, K, pairs * ksplit);
  if (lds > 160 * 1024) return -1;
  const int all_pairs = inner / 16;
  dim3 grid((all_pairs + pairs - 1) / pairs), block(pairs * ksplit * QIL_WAVE);
#define QIL_GATED_CASE(OUT, SILU)                                                                                       \
  {                                                                                                                  \
    auto kernel = gemm_bf16_gated_kernel<OUT, SILU>;                                                                 \
    static size_t granted = 0;                                                                                       \
    if (lds > 64 * 1024 && lds > granted) {                                                                          \
      hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds); \
      if (e != hipSuccess) return (int)e;                                                                            \
      granted = lds;                                                                                                 \
    }                                                                                                                \
    hipLaunchKernelGGL(kernel, grid, block, lds, s, (const bf16_t*)A, (const bf16_t*)W, (OUT*)out, M, inner, K, ksplit, interleaved, fn, \
                       NormedA());                                                                                   \
  }
  const bool silu = act == QIL_ACT_SILU;
  if (out_dtype == QIL_F32) {
    if (silu) QIL_GATED_CASE(float, true) else QIL_GATED_CASE(float, false)
  } else {
    if (silu) QIL_GATED_CASE(bf16_t, true) else QIL_GATED_CASE(bf16_t, false)
  }
#undef QIL_GATED_CASE
  QIL_RETURN_LAUNCH_STATUS();
}

// 1 if qil_gemm_bf16_gated_normed takes these sizes.
extern "C" int qil_gemm_bf16_gated_normed_takes(int M, int inner, int K) {
  int pairs, ksplit;
  return gated_plan(nullptr, nullptr, M, inner, K, &pairs, &ksplit) && M <= 2 * pairs * ksplit &&
         gated_lds(M, K, pairs * ksplit) + 16 * sizeof(float) <= 160 * 1024;
}

// out bfloat16 [M, inner] = silu(A gate^T) * (A up^T) for W with gate and up rows in turns of 16, A the norm of the float32 stream [M, K]
// (round, then the weight), made from its sums of squares in pieces as qil_gemm_bf16_normed does.
extern "C" int qil_gemm_bf16_gated_normed(const float* stream, const float* weight, const float* squares, int pieces, float eps,
                                          const void* W, void* out, int M, int inner, int K, hipStream_t s) {
  if (M == 0 || inner == 0) return 0;
  int pairs, ksplit;
  if (!qil_gemm_bf16_gated_normed_takes(M, inner, K) || !gated_plan(nullptr, W, M, inner, K, &pairs, &ksplit) || pieces < 1 ||
      (((uintptr_t)stream | (uintptr_t)weight) % 16))
    return -1;
  const NormedA normed{stream, weight, squares, pieces, eps};
  const size_t lds = gated_lds(M, K, pairs * ksplit) + 16 * sizeof(float);
  auto kernel = gemm_bf16_gated_kernel<bf16_t, true, true>;
  static size_t granted = 0;
  if (lds > 64 * 1024 && lds > granted) {
    const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
    granted = lds;
  }
  const int all_pairs = inner / 16;
  hipLaunchKernelGGL(kernel, dim3((all_pairs + pairs - 1) / pairs), dim3(pairs * ksplit * QIL_WAVE), lds, s, (const bf16_t*)nullptr,
                     (const bf16_t*)W, (bf16_t*)out, M, inner, K, ksplit, 1, GateFn{QIL_ACT_SILU, 0.f, 1.f}, normed);
  QIL_RETURN_LAUNCH_STATUS();
}

// silu(A W[:inner]^T) * (A W[inner:]^T)
extern "C" int qil_gemm_bf16_gated(const void* A, const void* W, void* out, int M, int inner, int K, int out_dtype,
                                   int pairs, int ksplit, int interleaved, hipStream_t s) {
  return qil_gemm_bf16_gated_act(A, W, out, M, inner, K, out_dtype, pairs, ksplit, interleaved, QIL_ACT_SILU, 0.f, 1.f, s);
}

// Shapes of the kernel that exist: code = MT * 100 + NT * 10 + UNROLL.
#define QIL_GEMM_SHAPES(X) \
  X(1, 1, 4) X(1, 1, 8) X(1, 2, 4) X(1, 2, 8) X(1, 4, 4) X(2, 1, 4) X(2, 1, 8) X(2, 2, 4) X(4, 1, 4) X(4, 1, 8) \
  X(4, 2, 4) X(4, 2, 2)

template <typename OUT>
static int launch_shape(int code, const bf16_t* A, const bf16_t* W, const float* bias, OUT* C, int M, int N, int K,
                        int splits, int chunk, hipStream_t s) {
#define X(MT, NT, UNROLL) \
  if (code == MT * 100 + NT * 10 + UNROLL) return launch_stream<MT, NT, UNROLL, OUT>(A, W, bias, C, M, N, K, splits, chunk, s);
  QIL_GEMM_SHAPES(X)
#undef X
  return -1;
}

// The plan for a product: kernel shape code and the number of K splits.
static void plan(int M, int N, int K, bool may_split, int* code, int* splits) {
  const int steps = (K + 31) / 32;
  const int mt = M <= 16 ? 1 : M <= 32 ? 2 : 4;
  const int column_blocks = (N + 127) / 128;
  int sp = 1;
  if (may_split) {
    // about three blocks per CU (256 CUs), at least 8 k steps per split, fewer splits for more rows
    const int most = 8;                                   // the consumer reads every partial
    sp = (3 * QIL_CUS + column_blocks - 1) / column_blocks;
    if (sp > most) sp = most;
    while (sp > 1 && steps / sp < 8) --sp;
    if (sp < 1) sp = 1;
    // up to 16 rows: of the splits the whole-line kernel takes (whole stages of 128 columns, at least LINES_DEPTH
    // of them; up to 32), the one with the least time by this count.  The blocks run in rounds of 256, one a CU; a
    // block's stage takes a unit of time while at most 160 blocks share the memory and more in proportion beyond
    // (measured: 160, 192, 256, 400 and 1,000 blocks stream equally well, 80 blocks take 50 % longer than 380); a
    // block's start (its slice of A, the first stages on their way) costs two units (the 1,187 column blocks of
    // Qwen3's logits: 226 us unsplit, 262 in four splits of 8 stages); every split adds 1.5 % for what the consumer
    // of the partial sums reads.
    if (M <= 16 && K % 128 == 0) {
      int fit = 0;
      double fit_time = 0;
      for (int c = 1; c <= 32; ++c) {
        if (K % (128 * c) || K / (128 * c) < LINES_DEPTH || lines_lds(M, K, c) > LINES_LDS_LIMIT) continue;
        const long blocks = (long)column_blocks * c, last = blocks % QIL_CUS;
        const int stages = K / (128 * c);
        double time = (double)(blocks / QIL_CUS) * (stages * 1.6 + 2.0);
        if (last) time += stages * std::max(1.0, last / 160.0) + 2.0;
        time *= 1.0 + 0.015 * c;
        if (!fit || time < fit_time) { fit = c; fit_time = time; }
      }
      if (fit) sp = fit;
    }
  }
  *code = mt * 100 + 10 + 4;
  *splits = sp;
}

// How many ways the product will be split over K when partial sums are allowed.
extern "C" int qil_gemm_bf16_splits(int M, int N, int K) {
  if (M > 16 && M <= CHUNKS_MOST_ROWS && K % 128 == 0 && K / 128 >= LINES_DEPTH) return chunks_splits(N, K);
  int code, splits;
  plan(M, N, K, true, &code, &splits);
  return splits;
}

// 1 if a product with 17 to 192 rows should run on the weight-streaming kernel here (K a multiple of 128 of at
// least 384, no bias; operands 16-byte aligned, which the call checks); products of up to 16 rows always do.
// 65 to 128 rows: only products of at most 64 column tiles (N <= 8192), which the split over K spreads over
// the CUs; measured at 128 rows and 8B layer sizes against the GPU BLAS: 21 us against 26 (q/k/v), 16 against
// 24 (attention output), 33 against 67 (down), but 57 against 49 for the 192 tiles of gate/up.
// 129 to 192 rows (a portion of 128 tokens beside decoded ones): at most 32 column tiles; at 160 rows 19 against
// 24 (attention output) and 39 against 60 (down), and level for the 48 tiles of q/k/v.
extern "C" int qil_gemm_bf16_streams(int M, int N, int K, int has_bias) {
  if (M <= 16) return 1;
  if (M > 64 && N > 64 * 16 * LINES_WAVES) return 0;
  if (M > 128 && N > 32 * 16 * LINES_WAVES) return 0;
  return chunks_takes(nullptr, nullptr, has_bias ? (const float*)1 : nullptr, M, N, K, 1);
}

// 1 if qil_gemm_bf16_unmerged takes these sizes (rows, output columns, heads, head size, K splits).
extern "C" int qil_gemm_bf16_unmerged_takes(int M, int N, int heads, int d, int splits) {
  const long K = (long)heads * d;
  if (M < 1 || M > 16 || N < 1 || d % 8 || splits < 1 || K > (1 << 30) || K % (128 * splits) || K / (128 * splits) < LINES_DEPTH)
    return 0;
  return lines_lds(M, (int)K, splits) <= LINES_LDS_LIMIT;
}

// C float32 [splits, M, N] = partial sums of merge(workspace) W^T, the merge being that of qil_attn_merge
// over a workspace laid out as qil_attn_rows_workspace describes (rows 0 .. M-1, no row index), made
// while the whole-line kernel stages A; K = heads * d.
extern "C" int qil_gemm_bf16_unmerged(const void* workspace, const int* positions, const void* W, void* C, int M, int N,
                                      int heads, int d, int window, int P, int parts, int splits, hipStream_t s) {
  if (M == 0 || N == 0) return 0;
  if (!qil_gemm_bf16_unmerged_takes(M, N, heads, d, splits) || parts < 1 || P < 0 || ((uintptr_t)W % 16) ||
      ((uintptr_t)workspace % 16))
    return -1;
  UnmergedA u;
  u.acc = (const float*)workspace;
  u.m = u.acc + (size_t)M * heads * parts * d;
  u.l = u.m + (size_t)M * heads * parts;
  u.positions = positions;
  u.heads = heads; u.d = d; u.parts = parts; u.P = P; u.window = window;
  u.part_keys = planned_keys(u.l, (size_t)M * heads * parts, P);
  const int status = launch_lines<float, 1>(nullptr, (const bf16_t*)W, (float*)C, M, N, heads * d, splits, s, u);
  if (status) return status;
  QIL_RETURN_LAUNCH_STATUS();
}

// 1 if qil_gemm_bf16_normed takes these sizes (rows, output columns, K, K splits).
extern "C" int qil_gemm_bf16_normed_takes(int M, int N, int K, int splits) {
  if (M < 1 || M > 16 || N < 1 || K % 8 || splits < 1 || K % (128 * splits) || K / (128 * splits) < LINES_DEPTH) return 0;
  return lines_lds(M, K, splits) <= LINES_LDS_LIMIT;
}

// C float32 [splits, M, N] = partial sums of rmsnorm(stream; weight, eps) W^T, the norm made while the whole-line
// kernel stages A from the float32 stream [M, K]; squares [pieces][M]: the rows' sums of squares in pieces.
extern "C" int qil_gemm_bf16_normed(const float* stream, const float* weight, const float* squares, int pieces, float eps,
                                    const void* W, void* C, int M, int N, int K, int splits, hipStream_t s) {
  if (M == 0 || N == 0) return 0;
  if (!qil_gemm_bf16_normed_takes(M, N, K, splits) || pieces < 1 ||
      (((uintptr_t)W | (uintptr_t)stream | (uintptr_t)weight) % 16))
    return -1;
  NormedA n;
  n.stream = stream; n.weight = weight; n.squares = squares; n.pieces = pieces; n.eps = eps;
  const int status = launch_lines<float, 2>(nullptr, (const bf16_t*)W, (float*)C, M, N, K, splits, s, UnmergedA(), n);
  if (status) return status;
  QIL_RETURN_LAUNCH_STATUS();
}

// out_dtype QIL_BF16: C bfloat16 [M, N], splits must be 1.  QIL_F32: C float32 [splits, M, N], the
// value being the sum over the first axis; bias (if any) requires splits == 1.
// shape: 0 = chosen here, else a code of QIL_GEMM_SHAPES; chunk: 0 = chosen here (tuning runs set both).
extern "C" int qil_gemm_bf16(const void* A, const void* W, const float* bias, void* C, int M, int N, int K,
                             int out_dtype, int splits, int shape, int chunk, hipStream_t s) {
  if (M == 0 || N == 0) return 0;
  if (K < 1 || splits < 1 || splits > 65535 || (splits > 1 && (out_dtype != QIL_F32 || bias))) return -1;
  int code = shape, planned;
  if (code == 0 || code == 1) {                              // 1: force the whole-line kernel (tuning runs)
    if (lines_takes(A, W, bias, M, N, K, splits)) {
      const int status = out_dtype == QIL_F32
                             ? launch_lines<float>((const bf16_t*)A, (const bf16_t*)W, (float*)C, M, N, K, splits, s)
                             : launch_lines<bf16_t>((const bf16_t*)A, (const bf16_t*)W, (bf16_t*)C, M, N, K, splits, s);
      if (status) return status;
      QIL_RETURN_LAUNCH_STATUS();
    }
    if (code == 1) return -1;
  }
  if (code == 0 || code == 2) {                              // 2: force the kernel that streams A (tuning runs)
    if (chunks_takes(A, W, bias, M, N, K, splits)) {
      const int status = out_dtype == QIL_F32
                             ? launch_chunks<float>((const bf16_t*)A, (const bf16_t*)W, (float*)C, M, N, K, splits, s)
                             : launch_chunks<bf16_t>((const bf16_t*)A, (const bf16_t*)W, (bf16_t*)C, M, N, K, splits, s);
      if (status) return status;
      QIL_RETURN_LAUNCH_STATUS();
    }
    if (code == 2) return -1;
  }
  if (!code) plan(M, N, K, false, &code, &planned);
  int status;
  if (out_dtype == QIL_F32)
    status = launch_shape<float>(code, (const bf16_t*)A, (const bf16_t*)W, bias, (float*)C, M, N, K, splits, chunk, s);
  else
    status = launch_shape<bf16_t>(code, (const bf16_t*)A, (const bf16_t*)W, bias, (bf16_t*)C, M, N, K, splits, chunk, s);
  if (status) return status;
  QIL_RETURN_LAUNCH_STATUS();
}
