// bfloat16 products of many rows (a prompt, a long portion of one):  C[M, N] = A[M, K] W[N, K]^T, float32
// accumulation, the matrix cores' work and no longer the memory's.
//
//  * A block makes 256 rows by 256 columns of C with eight waves, two a SIMD, each 128 rows by 64 columns with its
//    sums in 128 registers: per 16 columns of K a wave reads four fragments of A and two of W from LDS for eight
//    products v_mfma_f32_32x32x16_bf16, three quarters of a fragment read for a product (the kernel for 33 to 256
//    rows, a wave 32 columns wide and all the rows, reads more than one).  Four waves of 128 x 128, one a SIMD with
//    256 accumulation registers, read half a fragment a product and were 2 % slower: with one wave a SIMD nobody
//    multiplies while a wave waits for the barrier.  The products that do not give every CU such a block have blocks
//    of 128 x 128, four waves of 64 x 64 (128 x 256 and 256 x 128 with four waves were never the best of 60 products
//    of 300 to 2,048 rows, nor 128 x 128 with eight waves of 64 x 32).
//  * A and W go from memory straight into LDS (global_load_lds_dwordx4), a stage of 32 columns of K at a time into a
//    ring of AHEAD + 3 stages: a load is 16 rows of 64 bytes, whole halves of memory's
//    lines, and every wave sends its share of a stage's loads.  (W straight into registers, which a wave that owns
//    its columns alone could do, is 64 cache accesses a load, one a lane, where these are 16: the cache then took
//    longer than the products.)
//    Place p of row r holds the columns 8 (p ^ ((r >> 2) & 3)) ..: a fragment read takes 16 rows at a time, rows four
//    apart lie 256 bytes apart, on the same banks, and turned so the 16 pieces fall on all 64 banks once.
//  * The loads are sent one or two at a time between the products: a wave that sends its eight in a row waits some
//    50 cycles for each, the cache's queue being full of the other waves' loads, and the matrix core waits with it
//    (a block of 128 stages of four waves took 93 us so and 76 with a load behind every fourth product; its
//    products alone take 65).  They go out in pairs, load i of an even stage and of the next: the two halves of the same 128-byte
//    lines, which the cache then asks of L2 once and not twice.
//  * A wave waits for its own loads by their number in flight, and one barrier a stage makes them everyone's.  The
//    barrier for the next stage stands between the two halves of a stage's products, so that the first fragments of
//    the next stage are read while the second half multiplies, and the matrix core does not wait at a stage's start;
//    the results leave through LDS as whole rows of 128 columns (a lane's own 8 bytes into 32 rows an instruction
//    took a tenth of a block's time).  A pair of stages' loads go out one to two stages before the barrier that
//    hands its first stage on (a ring
//    of four stages with every load a stage later gave the same times: what the blocks wait for when every CU has
//    one is not the latency of a load).  A block of 128 x 128 alone on its CU is another matter: a stage is 256 cycles
//    of products, three of them are not a load's latency, and with the pairs six stages ahead (nine stages in LDS) 643
//    rows of 4,096 x 1,024 take 12.4 us and not 14.1, 1,000 rows 12.6 and not 14.1; two blocks a CU need no more than two.
//  * More rows than a block's are blocks of rows over the same W, which then comes from L2: the blocks of one XCD
//    (every eighth of the grid) take a run of consecutive pieces of work, numbered in patches of 8 row blocks by 4
//    column blocks, so that the 32 blocks that run together on an XCD read 12 different bands of A and W and not 33
//    (8,192 rows by 24,576 columns: 1.42 ms, 1.72 with the row blocks of one column block numbered through).  The
//    XCDs, and on an XCD the row blocks of a patch, begin at different stages of K and wrap round: blocks that go
//    in step ask for the same narrow band of every row, 8 KB apart, at the same time (gate/up at 2,048 rows with
//    every block of an XCD in step: 283 us on zeros and 326 on random operands; the row blocks apart: 259 and 316;
//    every block apart, which gives up the sharing of A as well: 274 and 338).
// Under load the time is the power's: with random operands the clock falls from 2.4 GHz to 1.45 to 1.7 when every CU
// multiplies (with zeros it stays above 2.1), so that a block's 177,000 cycles, of which the products are 131,000,
// take 105 to 125 us and not 75.
// Takes N a multiple of 32, K a multiple of 64 with at least 4 stages a split, 16-byte aligned operands of less than
// 4 GB each.
#include <algorithm>

#include "common.h"
#include "gated_act.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

#define WIDE_STAGE 32                                      // columns of K a stage: rows of 64 bytes
#define WIDE_ROW_BYTES (WIDE_STAGE * 2)
#define WIDE_XCDS 8
#define WIDE_SPLIT_COLUMNS 1024                            // fewest columns of a product of many rows that is left as partial sums
#define WIDE_HOST_US 24.0                                  // products of at most this time by wide_us are not the BLAS's ...
#define WIDE_GRAPH_ROWS 512                                // ... but up to so many rows, which a graph may replay,
#define WIDE_LEVEL_US 3.0                                  // only those within so much of its time on the GPU

// RT, CT: tiles of 32 rows and of 32 columns of a wave; DOWN, ACROSS: the block's waves above each other and side by side;
// AHEAD: stages (even) that a pair's loads go out ahead.  OUT: bf16_t or float (the result; with splits of K float32 partial sums [split][M][N]).  GATED (one split): W holds gate and up rows in turns of 16, a tile of 32 columns is 16
// of each, and C [M, N / 2] gets act(gate, up) (gated_act.h; qil/model.py:71), both still in float32.
template <typename OUT, int RT, int CT, int DOWN, int ACROSS, int AHEAD, int GATED>
__global__ void __launch_bounds__(DOWN * ACROSS * QIL_WAVE, RT * CT <= 4 && AHEAD == 2 ? 2 : 1)
gemm_bf16_wide_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, OUT* __restrict__ C, int M_all, int N, int K,
                      int stages, int col_blocks, int row_blocks, int splits, int patch_rows, int patch_cols, GateFn fn) {
  constexpr int WAVES = DOWN * ACROSS;
  constexpr int ROWS = 32 * RT * DOWN, TILE = 32 * CT * ACROSS;            // rows and columns of C a block
  constexpr int A_BYTES = ROWS * WIDE_ROW_BYTES, SLOT = A_BYTES + TILE * WIDE_ROW_BYTES;
  constexpr int A_LOADS = ROWS / 16 / WAVES, W_LOADS = TILE / 16 / WAVES;
  constexpr int LOADS = A_LOADS + W_LOADS;                 // a wave's loads a stage: those of A, then those of W
  constexpr int RING = AHEAD + 3;
  static_assert(LOADS % 2 == 0 && ROWS % (16 * WAVES) == 0 && TILE % (16 * WAVES) == 0, "whole loads, half of them in each half of a stage");
  static_assert(CT >= 2 && LOADS % 2 == 0 && 2 * ((LOADS / 2 + RT - 1) / RT) <= CT, "a load and a read a product at most");
  extern __shared__ __align__(1024) unsigned char ring[];  // a stage: the block's rows of A, then those of W, 64 bytes each
  const int lane = threadIdx.x & (QIL_WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / QIL_WAVE);
  // The piece of work.  XCD x (blocks x, x + 8, ...) takes the pieces x * per .. (x + 1) * per - 1, and the pieces are
  // numbered patch by patch: a patch is patch_rows row blocks by patch_cols column blocks, about as many as an XCD
  // has CUs, so that the blocks that run together on an XCD read few different rows of A and W.  Patches at the
  // edges have pieces that are no work.
  const int xcd = blockIdx.x % WIDE_XCDS, per = gridDim.x / WIDE_XCDS;
  const int item = xcd * per + blockIdx.x / WIDE_XCDS;
  const int in_patch = patch_rows * patch_cols;
  const int patches_down = (row_blocks + patch_rows - 1) / patch_rows, patches_across = (col_blocks + patch_cols - 1) / patch_cols;
  const int patch = item / in_patch, within = item % in_patch;
  const int split = patch / (patches_down * patches_across), patch_at = patch % (patches_down * patches_across);
  const int row_block = (patch_at % patches_down) * patch_rows + within % patch_rows;
  const int column_block = (patch_at / patches_down) * patch_cols + within / patch_rows;
  if (split >= splits || row_block >= row_blocks || column_block >= col_blocks) return;
  const int row0 = row_block * ROWS, M = min(M_all - row0, ROWS);
  const int n0 = column_block * TILE;
  const size_t k_begin = (size_t)split * stages * WIDE_STAGE;
  // the stage of K at which the block begins (even: a pair of stages stays the two halves of a line): its own for
  // every XCD and every row block of a patch
  const int turned = (int)((long)(xcd * patch_rows + within % patch_rows) * stages / (WIDE_XCDS * patch_rows)) & ~1;
  const int last = stages - 1;

  // Loads: a load is 16 rows of 64 bytes; lane = (row lane / 4, place lane % 4), and place p of row r takes piece
  // p ^ ((r >> 2) & 3) = p ^ ((lane >> 4) & 3).  Wave w brings the rows 16 A_LOADS w .. of A and 16 W_LOADS w .. of W.
  // Rows past the last repeat it: their results are not stored.
  const char* a_from = reinterpret_cast<const char*>(A + (size_t)row0 * K + k_begin);
  const char* w_from = reinterpret_cast<const char*>(W + k_begin);
  const uint32_t piece_bytes = (uint32_t)((lane & 3) ^ ((lane >> 4) & 3)) << 4;
  uint32_t row_bytes[LOADS];
#pragma unroll
  for (int i = 0; i < A_LOADS; ++i)
    row_bytes[i] = (uint32_t)min(16 * (A_LOADS * wave + i) + (lane >> 2), M - 1) * (uint32_t)K * 2 + piece_bytes;
#pragma unroll
  for (int i = 0; i < W_LOADS; ++i)
    row_bytes[A_LOADS + i] = (uint32_t)min(n0 + 16 * (W_LOADS * wave + i) + (lane >> 2), N - 1) * (uint32_t)K * 2 + piece_bytes;
  const uint32_t ring_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)ring;
  // Load i of a stage, as instructions: the memory's address is a scalar base and the lane's 32-bit offset, so that a
  // stage costs no vector arithmetic (the compiler adds 64-bit vector addresses for its own form of this load).  M0,
  // which holds the place in LDS, is written here behind the compiler's back: nothing else in this kernel uses it
  // (LDS reads and writes need no M0 on this hardware, and there is no other load into LDS).
  auto load = [&](int i, int stage, int slot) __attribute__((always_inline)) {
    const int k_stage = stage + turned < stages ? stage + turned : stage + turned - stages;
    const char* at = (i < A_LOADS ? a_from : w_from) + (size_t)k_stage * WIDE_ROW_BYTES;
    const uint32_t to = ring_at + slot * SLOT +
                        (i < A_LOADS ? (A_LOADS * wave + i) * 1024 : A_BYTES + (W_LOADS * wave + i - A_LOADS) * 1024);
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(row_bytes[i]), "s"(at), "s"(to) : "memory");
  };

  // Fragments: the wave's 32 RT rows of A and 32 CT columns of W, in tiles of 32; lane = (row lane % 32, half lane / 32)
  // wants piece 2 ks + half of its row, at place (2 ks + half) ^ ((row >> 2) & 3).
  const int l32 = lane & 31, half = lane >> 5;
  const uint32_t a_rows = (wave / ACROSS) * (32 * RT) * WIDE_ROW_BYTES, w_rows = A_BYTES + (wave % ACROSS) * (32 * CT) * WIDE_ROW_BYTES;
  uint32_t read_at[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) read_at[ks] = l32 * WIDE_ROW_BYTES + (((2 * ks + half) ^ ((l32 >> 2) & 3)) << 4);
  bf16x8 af[2][RT], wf[2][CT];
  f32x16 acc[RT][CT];                                      // [tile of rows][tile of columns]
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  // Load i of an even stage and of the stage after it, one behind the other: the two halves of the same 128-byte
  // lines, of which the cache then asks L2 once (asked a stage apart, each half cost a whole line, and with every
  // CU at work L2 was busy 93 % of the time).
  auto load_both = [&](int i, int even_stage) __attribute__((always_inline)) {
    load(i, min(even_stage, last), even_stage % RING);
    load(i, min(even_stage + 1, last), (even_stage + 1) % RING);
  };
  // The products of a tile of rows with the wave's tiles of columns, 16 columns of K, and what goes out meanwhile: the
  // reads of this tile's share of the other 16 columns' fragments, and this tile's share of the `doubles` double
  // loads `begin` .. of a later pair of stages.
  auto part = [&](int ks, int i, int read_slot, int begin, int doubles, int pair_stage) __attribute__((always_inline)) {
    const int other = ks ^ 1;
    const unsigned char* at = ring + read_slot * SLOT + read_at[other];
    const int first = doubles * i / RT, loads = 2 * (doubles * (i + 1) / RT - first);
    const int w_first = CT * i / RT, w_reads = CT * (i + 1) / RT - w_first;      // at most CT loads, at most CT - 1 reads of W
    // a product, and before it one of the reads and one of the loads: the order is the one written here
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      if (j == 0) af[other][i] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(at + a_rows + i * 2048));
      if (j >= 1 && j <= w_reads)
        wf[other][w_first + j - 1] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(at + w_rows + (w_first + j - 1) * 2048));
      if (j < loads) {
        const int stage = pair_stage + (j & 1);
        load(begin + first + j / 2, min(stage, last), stage % RING);
      }
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[ks][j], af[ks][i], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // Stage s lies in place s % RING.  The loads of the stages a + AHEAD and a + AHEAD + 1 (a even) go out as HALF double
  // loads in the second half of stage a - 1, behind the barrier that frees the place of stage a - 2, and HALF in the first
  // half of stage a; the barrier in the middle of a stage waits for the next stage's loads, behind which come one load
  // (the last of the odd stage of the same pair) or none of that pair, and the pairs after it.  Loads past the last stage bring the last one
  // again, into a place nobody reads any more, so that these counts hold at every stage.
  constexpr int HALF = LOADS / 2;
#pragma unroll
  for (int pair = 0; pair < AHEAD; pair += 2)
#pragma unroll
    for (int i = 0; i < LOADS; ++i) load_both(i, pair);
#pragma unroll
  for (int i = 0; i < HALF; ++i) load_both(i, AHEAD);
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(1 + LOADS * (AHEAD - 2) + 2 * HALF) : "memory");
#pragma unroll
  for (int t = 0; t < RT; ++t)
    af[0][t] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(ring + read_at[0] + a_rows + t * 2048));
#pragma unroll
  for (int t = 0; t < CT; ++t)
    wf[0][t] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(ring + read_at[0] + w_rows + t * 2048));
  for (int even = 0; even < stages; even += 2) {
    __builtin_amdgcn_sched_barrier(0);
    // the even stage: its first 16 columns multiply while the fragments of the second are read ...
#pragma unroll
    for (int i = 0; i < RT; ++i) part(0, i, even % RING, HALF, HALF, even + AHEAD);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(LOADS * AHEAD) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    // ... and its second 16 columns while the first fragments of the odd stage are read (behind the last stage: what
    // nobody multiplies)
#pragma unroll
    for (int i = 0; i < RT; ++i) part(1, i, (even + 1) % RING, 0, 0, 0);
    // the odd stage (the stages of a block are an even number)
#pragma unroll
    for (int i = 0; i < RT; ++i) part(0, i, (even + 1) % RING, 0, 0, 0);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(1 + LOADS * (AHEAD - 2)) : "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < RT; ++i) part(1, i, (even + 2) % RING, 0, HALF, even + AHEAD + 2);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // the loads past the end, into LDS

  // acc[i][j][e]: row 32 RT (wave / ACROSS) + 32 i + l32, column 32 CT (wave % ACROSS) + 32 j + 8 (e / 4) + 4 half + e % 4 of
  // the block.  Stored from here a lane would write 8 bytes into each of 16 places of its row, an instruction into 32
  // rows: 64 such instructions took a wave 15,000 to 28,000 cycles, a tenth of the block's time.  So a tile of 32
  // rows goes through LDS (the ring is done with; every wave has a corner of its own), and comes back as whole rows:
  // a lane stores 16 bytes, an instruction several rows of the wave's columns.
  asm volatile("s_barrier" ::: "memory");
  constexpr int KEPT = GATED ? 16 : 32;                    // columns of the result a tile of 32 columns of the product
  constexpr int ROW_BYTES = KEPT * CT * (int)sizeof(OUT) + 16;   // 16 more: the rows of a column start on different banks
  unsigned char* corner = ring + wave * (32 * ROW_BYTES);
  const int width = GATED ? N / 2 : N;                     // of a row of C
  const int first_column = (n0 + (wave % ACROSS) * (32 * CT)) / (GATED ? 2 : 1);
  OUT* out = C + ((size_t)split * M_all + row0) * width + first_column;
  constexpr int PIECES = KEPT * CT * (int)sizeof(OUT) / 16;  // 16-byte pieces of a row: 4 to 32
  const int piece = lane % PIECES, piece_row = lane / PIECES;
  const bool piece_in = first_column + (piece + 1) * (16 / (int)sizeof(OUT)) <= width;
#pragma unroll
  for (int i = 0; i < RT; ++i) {
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int g = 0; g < (GATED ? 2 : 4); ++g) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (GATED != QIL_UNGATED) {                           // columns 0-15 of a tile are gates, 16-31 the ups that belong to them
            v[e] = gate_by<GATED == QIL_GATED_SILU>(acc[i][j][4 * g + e], acc[i][j][4 * (g + 2) + e], fn);
          } else {
            v[e] = acc[i][j][4 * g + e];
          }
        }
        unsigned char* to = corner + l32 * ROW_BYTES + (KEPT * j + 8 * g + 4 * half) * (int)sizeof(OUT);
        if constexpr (sizeof(OUT) == 4) *reinterpret_cast<float4*>(to) = make_float4(v[0], v[1], v[2], v[3]);
        else *reinterpret_cast<uint2*>(to) = make_uint2(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]));
      }
    // the wave's own writes, read by itself: LDS takes a wave's instructions in order
#pragma unroll
    for (int r = 0; r < 32; r += QIL_WAVE / PIECES) {
      const int row = r + piece_row, m = (wave / ACROSS) * (32 * RT) + 32 * i + row;
      const uint4 v = *reinterpret_cast<const uint4*>(corner + row * ROW_BYTES + piece * 16);
      if (m < M && piece_in) *reinterpret_cast<uint4*>(reinterpret_cast<unsigned char*>(out + (size_t)m * width) + piece * 16) = v;
    }
  }
}

static bool wide_takes(int M, int N, int K, int splits) {
  if (M < 1 || N < 32 || N % 32 || K % (2 * WIDE_STAGE) || splits < 1) return false;
  if ((size_t)M * K * 2 >= ((size_t)1 << 32) || (size_t)N * K * 2 >= ((size_t)1 << 32)) return false;
  const int pairs = K / (2 * WIDE_STAGE);                  // a split is whole pairs of stages: whole 128-byte lines
  return pairs % splits == 0 && pairs / splits >= 2;
}

// The shapes of a block: 256 x 256 of C, 128 x 128 with two blocks a CU, and 128 x 128 with the whole LDS as its ring
// (one block a CU: what a CU has in flight is then the same as with two, for products that have no second block for it).
enum { WIDE_256 = 0, WIDE_128 = 1, WIDE_128_DEEP = 2 };

// How a product's pieces of work lie in its grid (the kernel's first lines): patches of row and column blocks, places
// without a piece at the patches' edges among them, and a run of as many places for each XCD.
struct WideGrid {
  int row_blocks, col_blocks, patch_rows, patch_cols, blocks;
};
static WideGrid wide_grid(int M, int N, int rows, int tile, int splits) {
  WideGrid g;
  g.row_blocks = (M + rows - 1) / rows;
  g.col_blocks = (N + tile - 1) / tile;
  g.patch_rows = std::min(g.row_blocks, 8);
  g.patch_cols = std::min(g.col_blocks, std::max(1, QIL_CUS / WIDE_XCDS / g.patch_rows));
  const int patches = ((g.row_blocks + g.patch_rows - 1) / g.patch_rows) * ((g.col_blocks + g.patch_cols - 1) / g.patch_cols) * splits;
  g.blocks = (patches * g.patch_rows * g.patch_cols + WIDE_XCDS - 1) / WIDE_XCDS * WIDE_XCDS;
  return g;
}

// A product's time by this count, us: a start and an end, rounds of blocks on the CUs times a stage's time, which grows
// with how many CUs work at once (memory, L2 and the clock are shared), and the partial sums out and in again at 5 TB/s.
// Fitted to products of 300 to 2,048 rows at 0.6B, 8B and 2,048 x 6,144 sizes with cold weights, which it meets to 15 %.
static double wide_us(int M, int N, int K, int splits, int shape) {
  const int edge = shape == WIDE_256 ? 256 : 128, slots = QIL_CUS * (shape == WIDE_128 ? 2 : 1);
  const WideGrid grid = wide_grid(M, N, edge, edge, splits);
  const long blocks = (long)grid.row_blocks * grid.col_blocks * splits;
  // One block a CU: the rounds of the XCD with the most pieces.  The first XCDs' places all hold one, and where the last
  // patches are nearly empty those are more than an eighth of the pieces (257 rows of 10,304 columns: 243 blocks, but 34
  // on XCDs of 32 CUs, 37 us where one round of K = 2,048 is 21).  Two a CU: what is left over runs alone, twice as fast.
  const long most = shape == WIDE_128 ? 0 : std::min<long>(blocks, grid.blocks / WIDE_XCDS);
  const long rounds = std::max((blocks + slots - 1) / slots, (most + slots / WIDE_XCDS - 1) / (slots / WIDE_XCDS));
  const double fill = (double)blocks / (rounds * slots);
  const double stage = shape == WIDE_256 ? 0.45 + 0.45 * fill : shape == WIDE_128 ? 0.30 + 0.23 * fill : 0.26;
  const double sums = splits > 1 ? 2.0 * splits * 4.0 * M * N / 5e6 : 0.0;
  return (shape == WIDE_256 ? 6.0 : 4.5) + rounds * ((double)K / WIDE_STAGE / splits) * stage + sums;
}

// The GPU BLAS's time for a product of up to 512 rows, us (fitted to 257 to 512 rows of 19 products from 512 x 4,096 to
// 12,288 x 2,048 with cold weights, which it meets to 24 %, 9 % on average), and the activation's behind it.
static double blas_us(int M, int N, int K, bool gated) {
  return 5.5 + 1.25e-9 * (2.0 * M * N * K) + 1.1 * K / 1024.0 + (gated ? 2.0 : 0.0);
}

// Whether a product of this time by the count above should not be the BLAS's.
static bool wide_wanted(int M, int N, int K, double us, bool gated) {
  return us <= WIDE_HOST_US && (M > WIDE_GRAPH_ROWS || us <= blas_us(M, N, K, gated) + WIDE_LEVEL_US);
}

template <typename OUT, int RT, int CT, int DOWN, int ACROSS, int AHEAD, int GATED>
static int wide_launch(const void* A, const void* W, void* C, int M, int N, int K, int splits, GateFn fn, hipStream_t s) {
  constexpr int ROWS = 32 * RT * DOWN, TILE = 32 * CT * ACROSS;
  const size_t lds = (size_t)(AHEAD + 3) * (ROWS + TILE) * WIDE_ROW_BYTES;
  auto kernel = gemm_bf16_wide_kernel<OUT, RT, CT, DOWN, ACROSS, AHEAD, GATED>;
  static bool granted = false;                             // per instantiation
  if (!granted) {
    hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
    granted = true;
  }
  const WideGrid g = wide_grid(M, N, ROWS, TILE, splits);
  hipLaunchKernelGGL(kernel, dim3(g.blocks), dim3(DOWN * ACROSS * QIL_WAVE), lds, s, (const bf16_t*)A, (const bf16_t*)W, (OUT*)C, M, N,
                     K, K / WIDE_STAGE / splits, g.col_blocks, g.row_blocks, splits, g.patch_rows, g.patch_cols, fn);
  QIL_RETURN_LAUNCH_STATUS();
}

template <int GATED>
static int wide_dispatch(int shape, const void* A, const void* W, void* C, int M, int N, int K, int out_dtype, int splits, hipStream_t s,
                         GateFn fn = {}) {
#define QIL_WIDE_CASE(SHAPE, RT, CT, DOWN, ACROSS, AHEAD)                                                             \
  case SHAPE:                                                                                                         \
    return out_dtype == QIL_F32 ? wide_launch<float, RT, CT, DOWN, ACROSS, AHEAD, GATED>(A, W, C, M, N, K, splits, fn, s) \
                                : wide_launch<bf16_t, RT, CT, DOWN, ACROSS, AHEAD, GATED>(A, W, C, M, N, K, splits, fn, s)
  switch (shape) {
    QIL_WIDE_CASE(WIDE_256, 4, 2, 2, 4, 2);
    QIL_WIDE_CASE(WIDE_128, 2, 2, 2, 2, 2);
    QIL_WIDE_CASE(WIDE_128_DEEP, 2, 2, 2, 2, 6);
  }
#undef QIL_WIDE_CASE
  return -1;
}

// The best shape at this number of splits.
static int wide_shape(int M, int N, int K, int splits) {
  double best = 1e30;
  int shape = WIDE_256;
  for (int one = WIDE_256; one <= WIDE_128_DEEP; ++one) {
    const double us = wide_us(M, N, K, splits, one);
    if (us < best) { best = us; shape = one; }
  }
  return shape;
}

extern "C" {

// 1 if qil_gemm_bf16_wide takes these sizes.
int qil_gemm_bf16_wide_takes(int M, int N, int K, int splits) { return wide_takes(M, N, K, splits); }

// The block's shape there (0: 256 x 256, 1: 128 x 128, 2: 128 x 128 with the long ring); a gated product has 2 * inner columns.
int qil_gemm_bf16_wide_shape(int M, int N, int K, int splits) { return wide_takes(M, N, K, splits) ? wide_shape(M, N, K, splits) : -1; }

// Splits of K with which a product of more than 256 rows should run here rather than in the GPU BLAS (1: a result of
// A's type; more, where `may_split` allows float32 partial sums, from 513 rows and 1,024 columns on, where there are no more
// columns than K); 0: the BLAS.  Fewer columns are not a stream's but factors that their consumer reads again and again (the 32
// columns of a state-space scan's B and C: left as partial sums of 4,096 rows of K, the scan's two passes over 2,048 rows took
// 96 and 54 us, with a bfloat16 result 51 and 40).
//
// Beyond 512 rows, where steps are launched kernel by kernel, what takes no more than WIDE_HOST_US by the count above stays
// here: the host spends 21 us on a library product and 7 on one of ours, and steps of such products wait for the host
// (prompts at 0.6B sizes, with the gated rule below, 530 rows 4.62 -> 2.69 ms, 1,000 rows 4.59 -> 3.26, 1,400 rows 4.93 ->
// 4.23, 2,048 rows, which the host does not hold up any more, 4.98 -> 5.04; at 8B and 2,048-wide sizes level).  On the GPU that costs nothing to 8 us a product (us here against there, 513 / 1,000
// rows: 4,096 x 1,024 12.5 / 13.8 against 13.3 / 13.7, 3,072 x 1,536 15.5 / 17.7 against 13.1 / 17.9, 2,048 x 2,048 18.6 / 19.5
// against 12.7 / 15.5, 1,024 x 2,048 18.5 / 18.7 against 10.7 / 11.3; 2,048 rows of 2,048 x 2,048 21.0 against 21.6).
//
// Up to 512 rows a graph may replay the step, where the host's time is nothing, and a step and its replay have to run the
// same kernels: there only products within WIDE_LEVEL_US of the library's time by its count (300 / 400 / 512 rows: 8,192 x
// 1,024 12.4 / 13.4 / 14.5 against 13.7 / 14.3 / 14.6, 4,096 x 1,024 11.9 / 12.0 / 12.1 against 10.2 / 10.7 / 10.8 and the
// library at 300; 5,120 x 2,048 19.8 / 22.5 against 21.3 / 23.2 at 400 / 512; the library's are 2,048 x 2,048 with 18.4 against 11.3, 1,024 x 1,024 with 11.2 against 8.7, 3,072 x 1,536 with 15.6
// against 13.3, 5,120 x 2,048 with 19.9 against 16.4 at 300), and no partial sums (with the norm behind them 2,048 x 2,048
// 19.3 against 15.1 at 400 rows, 1,024 x 1,024 13.2 against 12.3).
//
// Longer products are the library's inside a model even where this kernel is ahead alone (4,096 x 12,288 in 4 splits, 643
// rows: 78 us against 92 with cold operands, but 21 us a layer behind in a prompt of 530 rows, whose norms then read the
// partial sums).
int qil_gemm_bf16_wide_splits(int M, int N, int K, int may_split) {
  int found = 0;
  double best = 1e30;
  for (int splits = 1; splits <= (may_split && M > WIDE_GRAPH_ROWS && K >= N && N >= WIDE_SPLIT_COLUMNS ? 8 : 1); ++splits) {
    if (!wide_takes(M, N, K, splits)) continue;
    const double us = wide_us(M, N, K, splits, wide_shape(M, N, K, splits));
    if (us <= best && wide_wanted(M, N, K, us, false)) { best = us; found = splits; }
  }
  return found;
}

// C = A[M, K] W[N, K]^T.  splits > 1: C float32 [splits][M][N] partial sums (out_dtype QIL_F32); splits == 1: C [M][N]
// of out_dtype.
int qil_gemm_bf16_wide(const void* A, const void* W, void* C, int M, int N, int K, int out_dtype, int splits, hipStream_t s) {
  if (M == 0 || N == 0) return 0;
  if (!wide_takes(M, N, K, splits) || ((uintptr_t)A | (uintptr_t)W | (uintptr_t)C) % 16) return -1;
  if ((splits > 1 && out_dtype != QIL_F32) || (out_dtype != QIL_F32 && out_dtype != QIL_BF16)) return -1;
  return wide_dispatch<QIL_UNGATED>(wide_shape(M, N, K, splits), A, W, C, M, N, K, out_dtype, splits, s);
}

// 1 if qil_gemm_bf16_wide_gated takes these sizes: those of the product with 2 * inner columns in one split.
int qil_gemm_bf16_wide_gated_takes(int M, int inner, int K) { return inner >= 16 && inner % 16 == 0 && wide_takes(M, 2 * inner, K, 1); }

// 1 if a gated product of more than 256 rows should run here: by the same rule, and two kernels become one (643 rows of
// 6,144 x 1,024 18.5 us, inside a prompt 22, against 18.9 and 4.4 for the activation; 2,048 rows 30.7 against 27.4 and 9.6, but a prompt of
// 2,048 rows 4.89 ms against 4.78, of 5,000 13.1 against 12.8; up to 512 rows inner 3,072 x 1,024 13.2 against 19.0 with the
// activation, 4,096 x 1,024 14.4 against 20.2, and the library's 1,024 x 2,048 with 19.6 against 13.9).
int qil_gemm_bf16_wide_gated_wanted(int M, int inner, int K) {
  return M > 256 && qil_gemm_bf16_wide_gated_takes(M, inner, K) &&
         wide_wanted(M, 2 * inner, K, wide_us(M, 2 * inner, K, 1, wide_shape(M, 2 * inner, K, 1)), true);
}

// out [M, inner] of out_dtype = act(A gate^T, A up^T) for W [2 inner, K] with gate and up rows in turns of 16; act, limit,
// alpha: a gate function of gated_act.h.
int qil_gemm_bf16_wide_gated_act(const void* A, const void* W, void* out, int M, int inner, int K, int out_dtype, int act,
                                 float limit, float alpha, hipStream_t s) {
  if (!gate_fn_known(act)) return -1;
  if (M == 0 || inner == 0) return 0;
  if (!qil_gemm_bf16_wide_gated_takes(M, inner, K) || ((uintptr_t)A | (uintptr_t)W | (uintptr_t)out) % 16 ||
      (out_dtype != QIL_F32 && out_dtype != QIL_BF16))
    return -1;
  const GateFn fn{act, limit, alpha};
  const int shape = wide_shape(M, 2 * inner, K, 1);
  return act == QIL_ACT_SILU ? wide_dispatch<QIL_GATED_SILU>(shape, A, W, out, M, 2 * inner, K, out_dtype, 1, s, fn)
                             : wide_dispatch<QIL_GATED_OTHER>(shape, A, W, out, M, 2 * inner, K, out_dtype, 1, s, fn);
}

// silu(A gate^T) * (A up^T)
int qil_gemm_bf16_wide_gated(const void* A, const void* W, void* out, int M, int inner, int K, int out_dtype, hipStream_t s) {
  return qil_gemm_bf16_wide_gated_act(A, W, out, M, inner, K, out_dtype, QIL_ACT_SILU, 0.f, 1.f, s);
}

}  // extern "C"
