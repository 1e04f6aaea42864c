// A few-row bfloat16 product that adds its result into the float32 residual stream:
//   stream[M, N] += A[M, K] W[N, K]^T,   M <= 16, float32 accumulation.
// A block owns `groups` groups of 16 (or 8, below) output columns and `ksplit` waves per group, which split K among themselves and
// add their float32 sums in LDS in wave order (the scheme of the gated kernel in gemm_bf16.hip): no partial sums in
// memory, every element of the stream is read, added to and written by one lane, after its sum is complete.  The
// kernel that follows finds the stream complete: it needs no sum over partial results, and the norm it would start
// with can be made by the product after it (gemm_bf16.hip, NormedA), for which this kernel leaves the rows' sums of
// squares in pieces: squares[piece][m] = sum over the columns of group `piece` of stream[m, .]^2.
// W and A both travel in whole cache lines (4 rows x 256 bytes a load), three stages of 128 columns ahead in
// registers, through buffers of the wave's own in LDS that turn them into matrix-core fragments (see the whole-line
// kernel in gemm_bf16.hip); A comes from L2.  K may be any length (the down product of a gated feed-forward).
// The same kernel makes the products whose bfloat16 result has to be whole (no consumer of partial sums behind them).
// Takes N a multiple of 16, K a multiple of 128 ksplit with at least 3 stages a wave, 16-byte aligned operands.
#include <algorithm>

#include "common.h"
#include "merge_parts.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

#define ADD_WAVES 8                                        // most waves of a block
#define ADD_DEPTH 3                                        // stages in flight per wave
#define ADD_LDS_LIMIT (160 * 1024)

// AROWS: rows of A kept (8 or 16).  COLS: columns of a group, 16 or 8 (the matrix cores then make every column twice and memory
// is read once: twice the groups, where those of 16 leave half of the CUs without a block).  INTO: the result goes into the
// stream; else out [M, N] of bfloat16 gets it (squares null).
template <int AROWS, bool INTO, int COLS = 16>
__global__ void __launch_bounds__(ADD_WAVES * QIL_WAVE, COLS == 8 ? 2 : AROWS == 8 ? 4 : 3)
gemm_bf16_add_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, float* __restrict__ stream,
                     bf16_t* __restrict__ out, float* __restrict__ squares, int M, int N, int K, int ksplit) {
  extern __shared__ __align__(16) bf16_t lds[];            // per wave: COLS x 256 bytes for W, AROWS x 256 for A
  constexpr int ALOADS = AROWS / 4, WLOADS = COLS / 4, PER_WAVE = (COLS + AROWS) * 128;
  const int lane = threadIdx.x & (QIL_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / QIL_WAVE);
  const int r = lane & 15, kb = lane >> 4;
  const int group = wave / ksplit, part = wave - group * ksplit;
  const int groups = blockDim.x / QIL_WAVE / ksplit;
  const int mine = blockIdx.x * groups + group;
  const bool stores = mine * COLS < N && (lane & 15) < COLS;
  const int n0 = min(mine, N / COLS - 1) * COLS;               // a group past the end repeats the last one and stores nothing
  const int cols = K / ksplit, k_begin = part * cols, stages = cols / 128;
  // Every wave walks its K range from a start of its own and wraps around: waves that all read the same columns
  // of their rows at the same time load a few memory channels only.
  const int turn = (n0 / COLS) % stages;
  auto column = [&](int stage) { const int st = stage + turn; return (st >= stages ? st - stages : st) * 128; };
  bf16_t* buffer = lds + wave * PER_WAVE;
  bf16_t* a_buffer = buffer + COLS * 128;

  // a load's address is a scalar base (the wave's rows and columns) and an offset of the lane's
  const int load_row = lane >> 4, piece = lane & 15;
  const char* w_base = reinterpret_cast<const char*>(W + (size_t)n0 * K + k_begin);
  const char* a_base = reinterpret_cast<const char*>(A + k_begin);
  const uint32_t w_offset = (uint32_t)load_row * (uint32_t)K * 2 + piece * 16;
  uint32_t a_offset[ALOADS];                               // (rows of A past the last read it again: rows of D never stored)
  int place[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int row = 4 * u + load_row;
    place[u] = row * 128 + ((piece ^ row) & 15) * 8;
    if (u < ALOADS) a_offset[u] = (uint32_t)min(row, M - 1) * (uint32_t)K * 2 + piece * 16;
  }
  u32x4 w0[WLOADS], w1[WLOADS], w2[WLOADS], a0[ALOADS], a1[ALOADS], a2[ALOADS];   // named, so that none is indexed at run time
  auto request = [&](u32x4 (&stage_w)[WLOADS], u32x4 (&stage_a)[ALOADS], int stage) {
    const size_t at = (size_t)column(stage) * 2;
#pragma unroll
    for (int u = 0; u < WLOADS; ++u) stage_w[u] = load_once(w_base + at + (size_t)(4 * u) * K * 2 + w_offset);
#pragma unroll
    for (int u = 0; u < ALOADS; ++u) stage_a[u] = *reinterpret_cast<const u32x4*>(a_base + at + a_offset[u]);
  };
  request(w0, a0, 0);
  request(w1, a1, 1);
  request(w2, a2, 2);

  // The cells of the stream that this lane will add to come in behind the first stages: read when the sums are there, they were one
  // more trip to memory at the kernel's end (with the barrier that the sums' own buffers save and the squares' shuffles: one row of 1,024 x
  // 3,072 5.3 -> 4.7 us, 8 rows 6.7 -> 5.3, 8 of 4,096 x 12,288 19.4 -> 18.0, 16 of 4,096 x 4,096 10.4 -> 9.1).
  float cell[4] = {0.f, 0.f, 0.f, 0.f};
  if (INTO)
#pragma unroll
    for (int i = 0; i < 4; ++i) cell[i] = stream[(size_t)min(4 * kb + i, M - 1) * N + n0 + (r & (COLS - 1))];

  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  const int a_row = r & (AROWS - 1), w_row = r & (COLS - 1);
  auto step = [&](u32x4 (&stage_w)[WLOADS], u32x4 (&stage_a)[ALOADS], int next, bool more) {
#pragma unroll
    for (int u = 0; u < WLOADS; ++u) *reinterpret_cast<u32x4*>(buffer + place[u]) = stage_w[u];
#pragma unroll
    for (int u = 0; u < ALOADS; ++u) *reinterpret_cast<u32x4*>(a_buffer + place[u]) = stage_a[u];
    if (more) request(stage_w, stage_a, next);
    __builtin_amdgcn_wave_barrier();                        // LDS operations of one wave complete in order: no wait
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      const u32x4 b = *reinterpret_cast<const u32x4*>(buffer + w_row * 128 + (((4 * s4 + kb) ^ w_row) & 15) * 8);
      const u32x4 a = *reinterpret_cast<const u32x4*>(a_buffer + a_row * 128 + (((4 * s4 + kb) ^ a_row) & 15) * 8);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0,
                                                    0, 0);
    }
    __builtin_amdgcn_wave_barrier();
  };
  int stage = 0;
  for (; stage + 6 <= stages; stage += 3) {                 // every stage here has a successor three ahead
    step(w0, a0, stage + 3, true);
    step(w1, a1, stage + 4, true);
    step(w2, a2, stage + 5, true);
  }
  const int left = stages - stage;                          // three to five stages: requests run out
  step(w0, a0, stage + 3, left > 3);
  step(w1, a1, stage + 4, left > 4);
  step(w2, a2, 0, false);
  if (left > 3) step(w0, a0, 0, false);
  if (left > 4) step(w1, a1, 0, false);

  // The waves' sums meet in LDS ([lane][4] floats, each wave's in its own buffer, which it has finished with); part 0 of
  // each group adds them in wave order; the lane that holds D[m = 4 kb + i][n = r] adds it into the stream.
  float* sums = reinterpret_cast<float*>(lds);
  *reinterpret_cast<f32x4*>(sums + wave * (PER_WAVE / 2) + lane * 4) = acc;
  __syncthreads();
  if (part == 0) {
    f32x4 total = {0.f, 0.f, 0.f, 0.f};
    for (int v = wave; v < wave + ksplit; ++v)              // fixed order
      total += *reinterpret_cast<const f32x4*>(sums + v * (PER_WAVE / 2) + lane * 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = 4 * kb + i;
      float value = 0.f;
      if (!INTO) {
        if (m < M && stores) out[(size_t)m * N + n0 + r] = f32_to_bf16(total[i]);
        continue;
      }
      if (m < M && stores) {
        value = cell[i] + total[i];
        stream[(size_t)m * N + n0 + r] = value;
      }
      if (squares) {                                        // the lanes of a row add their squares: one order for all
        float square = value * value;
        square += lane_move<0xB1>(square);               // quads (1, 0, 3, 2): the neighbour
        square += lane_move<0x4E>(square);               // quads (2, 3, 0, 1)
        square += lane_move<0x141>(square);              // halves of 16 mirrored: the other quad, whose lanes agree by now
        if (COLS == 16) square += lane_move<0x140>(square);          // 16 mirrored: the other half
        if (r == 0 && m < M && stores) squares[(size_t)mine * M + m] = square;
      }
    }
  }
}

// The same behind split-context attention, few rows: A [M, K = heads * d] is merged from the attention's parts (merge_parts.h) while W is
// on its way.  A block owns 8 columns and 8 waves share K, whose STAGES stages of 128 columns a wave are all asked for at once; every
// block merges all of its rows (from L2).  With the stream complete behind it and its squares left, the next product makes the second
// norm of a layer itself: one kernel less.  What bounds it is the chain parts, merge, products, sums, stream.
template <int STAGES>
__global__ void __launch_bounds__(ADD_WAVES * QIL_WAVE)
gemm_bf16_merge_add_kernel(const bf16_t* __restrict__ W, float* __restrict__ stream, float* __restrict__ squares, int M, int N, int K,
                           UnmergedA unmerged) {
  extern __shared__ __align__(16) bf16_t lds[];            // A [8][K + 8], then 8 x 256 bytes of W a wave
  constexpr int COLS = 8, A_ROWS = 8, THREADS = ADD_WAVES * QIL_WAVE, PER_WAVE = COLS * 128;
  const int lane = threadIdx.x & (QIL_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / QIL_WAVE);
  const int r = lane & 15, kb = lane >> 4, load_row = lane >> 4, piece = lane & 15;
  const int n0 = blockIdx.x * COLS, k_begin = wave * STAGES * 128, row_width = K + 8;
  bf16_t* buffer = lds + A_ROWS * row_width + wave * PER_WAVE;
  const int pieces = K / 8, all = M * pieces, P = merge_part_keys(unmerged);
  MergeParts<8, 4> parts;
  int idx = threadIdx.x, m0, c0;
  auto ask = [&](int of) __attribute__((always_inline)) {
    m0 = of / pieces;
    c0 = (of - m0 * pieces) * 8;
    merge_ask(unmerged, P, m0, c0, parts);
  };
  auto put = [&]() __attribute__((always_inline)) {
    float v[8];
    merge_finish(unmerged, P, m0, c0, parts, v);
    *reinterpret_cast<uint4*>(lds + m0 * row_width + c0) =
        make_uint4(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7]));
  };
  ask(min(idx, all - 1));
  __builtin_amdgcn_sched_barrier(0);
  u32x4 w[STAGES][2];
#pragma unroll
  for (int st = 0; st < STAGES; ++st)
#pragma unroll
    for (int u = 0; u < 2; ++u)
      w[st][u] = load_once(W + (size_t)(n0 + 4 * u + load_row) * K + k_begin + st * 128 + piece * 8);
  float cell[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) cell[i] = stream[(size_t)min(4 * kb + i, M - 1) * N + n0 + (r & (COLS - 1))];
  __builtin_amdgcn_sched_barrier(0);
  parts.arrived();
  if (idx < all) put();
  for (idx += THREADS; idx < all; idx += THREADS) {
    ask(idx);
    put();
  }
  __syncthreads();

  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  const int w_row = r & (COLS - 1);
  const bf16_t* a_row = lds + (r & (A_ROWS - 1)) * row_width + k_begin + kb * 8;     // (rows past M: products that are never stored)
#pragma unroll
  for (int st = 0; st < STAGES; ++st) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int row = 4 * u + load_row;
      *reinterpret_cast<u32x4*>(buffer + row * 128 + ((piece ^ row) & 15) * 8) = w[st][u];
    }
    __builtin_amdgcn_wave_barrier();                        // LDS operations of one wave complete in order: no wait
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) {
      const u32x4 b = *reinterpret_cast<const u32x4*>(buffer + w_row * 128 + (((4 * s4 + kb) ^ w_row) & 15) * 8);
      const u32x4 a = *reinterpret_cast<const u32x4*>(a_row + st * 128 + s4 * 32);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), acc, 0, 0, 0);
    }
    __builtin_amdgcn_wave_barrier();
  }
  float* sums = reinterpret_cast<float*>(lds + A_ROWS * row_width);      // the waves' sums, each in its own buffer
  *reinterpret_cast<f32x4*>(sums + wave * (PER_WAVE / 2) + lane * 4) = acc;
  __syncthreads();
  if (wave == 0) {
    f32x4 total = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int v = 0; v < ADD_WAVES; ++v) total += *reinterpret_cast<const f32x4*>(sums + v * (PER_WAVE / 2) + lane * 4);   // fixed order
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int m = 4 * kb + i;
      const bool stores = m < M && r < COLS;
      const float value = stores ? cell[i] + total[i] : 0.f;
      if (stores) stream[(size_t)m * N + n0 + r] = value;
      float square = value * value;
      square += lane_move<0xB1>(square);
      square += lane_move<0x4E>(square);
      square += lane_move<0x141>(square);
      if (stores && r == 0) squares[(size_t)blockIdx.x * M + m] = square;
    }
  }
}

static size_t add_lds_bytes(int M, int waves, int cols = 16) {
  return (size_t)waves * (cols + (M <= 8 ? 8 : 16)) * 128 * sizeof(bf16_t);   // also holds the waves' sums (1 KB a wave)
}

// Groups of 8 columns instead of 16: up to 8 rows of products whose groups of 16 fill at most half of the CUs with a block each
// (a CU draws 36 GB/s at most): 1,024 x 3,072, one row, 6.4 -> 5.8 us inside a step (64 blocks of 98 KB, 128 of 49), 2,048 x 6,144,
// 8 rows, 10.7 -> 9.2.
static bool add_narrow(int M, int N, int K) {
  return M <= 8 && N >= 512 && N <= 16 * QIL_CUS / 2 && K % 1024 == 0 && K / 1024 >= ADD_DEPTH;
}

// Waves a group and groups a block for these sizes; false if the kernel does not take them.
static bool add_plan(int M, int N, int K, int* groups, int* ksplit) {
  if (M < 1 || M > 16 || N < 16 || N % 16 || K < 128 * ADD_DEPTH || K % 128 || K > 1 << 27) return false;     // (a lane's offset: 32 bits)
  const int all_groups = N / 16;
  int best_groups = 0, best_ksplit = 0;
  double best_cost = 0;
  for (int ks = 8; ks >= 1; ks /= 2) {
    if (K % (128 * ks) || K / (128 * ks) < ADD_DEPTH) continue;
    for (int gb = ADD_WAVES / ks; gb >= 1; --gb) {
      const size_t lds = add_lds_bytes(M, gb * ks);
      // blocks of a CU at a time: by LDS and by the wave slots its registers leave (16 for up to 8 rows, 12 beyond);
      // rounds of the whole chip; a CU's waves keep memory busy when there are 8 or more of them
      const long slots = M <= 8 ? 16 : 12;
      const long together = std::max<long>(1, std::min<long>((long)(ADD_LDS_LIMIT / lds), slots / (gb * ks)));
      const long blocks = (all_groups + gb - 1) / gb;
      const long rounds = (blocks + QIL_CUS * together - 1) / (QIL_CUS * together);
      const long busy = std::min<long>(8, std::min<long>(together, (blocks + QIL_CUS - 1) / QIL_CUS) * gb * ks);
      const double cost = (double)rounds * gb * 8.0 / (double)busy + 0.05 * rounds;
      if (!best_groups || cost < best_cost) { best_groups = gb; best_ksplit = ks; best_cost = cost; }
    }
  }
  if (!best_groups) return false;
  *groups = best_groups;
  *ksplit = best_ksplit;
  return true;
}

extern "C" {

// 1 if qil_gemm_bf16_add takes these sizes.
int qil_gemm_bf16_add_takes(int M, int N, int K) {
  int groups, ksplit;
  return add_plan(M, N, K, &groups, &ksplit);
}

}  // extern "C"

template <bool INTO>
static int add_launch(const void* A, const void* W, float* stream, void* out, float* squares, int M, int N, int K, int groups,
                      int ksplit, hipStream_t s, bool narrow = false) {
  if (M == 0 || N == 0) return 0;
  if (((uintptr_t)A | (uintptr_t)W | (uintptr_t)stream) % 16) return -1;
  int planned_groups, planned_ksplit;
  if (!add_plan(M, N, K, &planned_groups, &planned_ksplit)) return -1;
  if (INTO && narrow) {
    hipLaunchKernelGGL((gemm_bf16_add_kernel<8, INTO, 8>), dim3(N / 8), dim3(ADD_WAVES * QIL_WAVE), add_lds_bytes(M, ADD_WAVES, 8), s,
                       (const bf16_t*)A, (const bf16_t*)W, stream, (bf16_t*)out, squares, M, N, K, ADD_WAVES);
    QIL_RETURN_LAUNCH_STATUS();
  }
  if (!groups) groups = planned_groups;
  if (!ksplit) ksplit = planned_ksplit;
  if (groups < 1 || ksplit < 1 || groups * ksplit > ADD_WAVES || K % (128 * ksplit) || K / (128 * ksplit) < ADD_DEPTH)
    return -1;
  const size_t lds = add_lds_bytes(M, groups * ksplit);
  dim3 grid((N / 16 + groups - 1) / groups), block(groups * ksplit * QIL_WAVE);
  if (M <= 8)
    hipLaunchKernelGGL((gemm_bf16_add_kernel<8, INTO>), grid, block, lds, s, (const bf16_t*)A, (const bf16_t*)W, stream,
                       (bf16_t*)out, squares, M, N, K, ksplit);
  else
    hipLaunchKernelGGL((gemm_bf16_add_kernel<16, INTO>), grid, block, lds, s, (const bf16_t*)A, (const bf16_t*)W, stream,
                       (bf16_t*)out, squares, M, N, K, ksplit);
  QIL_RETURN_LAUNCH_STATUS();
}

extern "C" {

// stream float32 [M, N] += A[M, K] W[N, K]^T.  squares: null, or float32 [N / 16][M] that gets the rows' sums of squares of
// the new stream in pieces of 16 columns.  groups, ksplit: 0 = chosen here (tuning runs and tests set them).
int qil_gemm_bf16_add(const void* A, const void* W, float* stream, float* squares, int M, int N, int K, int groups,
                      int ksplit, hipStream_t s) {
  return add_launch<true>(A, W, stream, nullptr, squares, M, N, K, groups, ksplit, s);
}

// The same in groups of 16 or 8 columns, whichever these sizes run better in.  squares: float32 [pieces][M]; pieces, the size
// of the caller's array, has to be what qil_gemm_bf16_add_pieces says (N / 16, or N / 8).
int qil_gemm_bf16_add_pieces(int M, int N, int K) { return add_narrow(M, N, K) ? N / 8 : N / 16; }
int qil_gemm_bf16_add_in_pieces(const void* A, const void* W, float* stream, float* squares, int pieces, int M, int N, int K,
                                hipStream_t s) {
  if (M == 0 || N == 0) return 0;
  if (pieces != qil_gemm_bf16_add_pieces(M, N, K)) return -1;
  return add_launch<true>(A, W, stream, nullptr, squares, M, N, K, 0, 0, s, add_narrow(M, N, K));
}

// 1 if a product of up to 16 rows whose result has to be whole and of bfloat16 should run here (qil_gemm_bf16_whole): where
// the whole-line kernel (gemm_bf16.hip), which can split K only into partial sums, is a block of 128 columns on each of few
// CUs.  us there and here, 8 rows: 3,072 x 1,536 10.0 / 6.1, 6,144 x 2,048 13.2 / 7.9, 12,288 x 2,048 16.5 / 10.9, 16,384 x
// 2,048 16.7 / 13.4, 32,768 x 2,048 22.9 / 23.2, 4,096 x 4,096 22.3 / 8.7, 2,048 x 6,144 70 / 10.7, 1,536 x 512 5.0 / 6.1.
// A K of an odd number of stages cannot be split over waves, and with no more groups of columns than CUs the plan then has
// fewer waves than that kernel's: 4,096 x 1,152 8.1 / 10.1, 1,024 x 3,200 17.6 / 22.4, 16 rows of 2,048 x 6,272 36.6 / 52.4;
// with more groups it is ahead (4,112 x 1,152 8.1 / 4.8), and so for up to 8 rows where K is too long for the whole-line
// kernel (1,024 x 4,480 50.7 / 30.5).
int qil_gemm_bf16_whole_takes(int M, int N, int K) {
  int groups, ksplit;
  if (N > 16384 || K < 1024 || !add_plan(M, N, K, &groups, &ksplit)) return 0;
  return ksplit > 1 || N > 16 * QIL_CUS || (M <= 8 && K > 4224);
}

// out bfloat16 [M, N] = A[M, K] W[N, K]^T, K split over a block's waves.
int qil_gemm_bf16_whole(const void* A, const void* W, void* out, int M, int N, int K, hipStream_t s) {
  return add_launch<false>(A, W, nullptr, out, nullptr, M, N, K, 0, 0, s);
}

// 1 if qil_gemm_bf16_unmerged_add takes these sizes: up to four rows and 16 parts in all, at most a block of 8 columns a CU, one to four
// stages a wave.  Every block merges all rows, which beyond that costs more than the norm's kernel: us a step of 28 layers with partial
// sums and a norm / so: 1 row of 100 keys 879 / 810, of 3,600 (16 parts) 968 / 903; 2 rows of 100 900 / 840, of 512 (4 parts each) 897 / 853, of
// 1,600 (8 parts) 939 / 897; 3 rows of 300 930 / 917, of 600 (4 parts) 932 / 917; 4 rows of 100 928 / 917, of 512 (4 parts) 951 / 937; but 4 of 2,000
// (8 parts) 1,038 / 1,057, 5 of 100 980 / 1,015, 8 of 300 999 / 1,042.  4,096 columns, two blocks a CU, 12 layers: 1 row of 100 keys 1,184 / 1,204, of
// 2,048 1,252 / 1,315, 4 of 100 1,260 / 1,371.
#define MERGE_ADD_ROWS 4
#define MERGE_ADD_PARTS 16
int qil_gemm_bf16_unmerged_add_takes(int M, int N, int heads, int d, int parts) {
  if (M < 1 || M > MERGE_ADD_ROWS || N < 8 || N % 8 || N > 8 * QIL_CUS || heads < 1 || d < 8 || d % 8 || heads > 65536 || d > 65536) return 0;
  const long K = (long)heads * d;
  return K % 1024 == 0 && K <= 4096 && parts >= 1 && (long)M * parts <= MERGE_ADD_PARTS;
}

// stream float32 [M, N] += merge(workspace) W^T, the workspace as qil_gemm_bf16_unmerged takes it; squares float32 [N / 8][M]: the rows'
// sums of squares of the new stream in pieces of 8 columns.
int qil_gemm_bf16_unmerged_add(const void* workspace, const int* positions, const void* W, float* stream, float* squares, int M, int N,
                               int heads, int d, int window, int P, int parts, hipStream_t s) {
  if (M == 0 || N == 0) return 0;
  if (!qil_gemm_bf16_unmerged_add_takes(M, N, heads, d, parts) || P < 0 || !squares ||
      (((uintptr_t)W | (uintptr_t)workspace | (uintptr_t)stream) % 16))
    return -1;
  const int K = heads * d;
  UnmergedA u;
  u.acc = (const float*)workspace;
  u.m = u.acc + (size_t)M * heads * parts * d;
  u.l = u.m + (size_t)M * heads * parts;
  u.positions = positions;
  u.heads = heads; u.d = d; u.parts = parts; u.P = P; u.window = window;
  u.part_keys = planned_keys(u.l, (size_t)M * heads * parts, P);
  const size_t lds = ((size_t)8 * (K + 8) + ADD_WAVES * 8 * 128) * sizeof(bf16_t);
#define QIL_MERGE_ADD(STAGES)                                                                                                    \
  {                                                                                                                              \
    auto kernel = gemm_bf16_merge_add_kernel<STAGES>;                                                                            \
    static bool granted = false;                             /* per instantiation */                                             \
    if (lds > 64 * 1024 && !granted) {                                                                                           \
      const hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);       \
      if (e != hipSuccess) return (int)e;                                                                                        \
      granted = true;                                                                                                            \
    }                                                                                                                            \
    hipLaunchKernelGGL(kernel, dim3(N / 8), dim3(ADD_WAVES * QIL_WAVE), lds, s, (const bf16_t*)W, stream, squares, M, N, K, u);  \
  }
  switch (K / 1024) {
    case 1: QIL_MERGE_ADD(1) break;
    case 2: QIL_MERGE_ADD(2) break;
    case 3: QIL_MERGE_ADD(3) break;
    default: QIL_MERGE_ADD(4)
  }
#undef QIL_MERGE_ADD
  QIL_RETURN_LAUNCH_STATUS();
}

}  // extern "C"
