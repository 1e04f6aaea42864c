// The tile kernel of attention_tile.hip for common cases, written without branches in the tile loop: bfloat16, head
// size exactly D (64 or 256; 128 goes on to attention_prompt.hip from here), a page size that is a power of two from
// 8 on, a block table of a sequence that fits in LDS.  Same block shape, same matrix-core formulation, same order of
// every sum, so a row gets bit for bit the result of the general kernel (qil/model.py:59-66 is the formula of both).
//
// What differs is the schedule:
//  * the sequence's block-table entries are copied to LDS once, so finding a page is an LDS read and
//    not a load that the K and V loads must wait for;
//  * while a tile is multiplied, the next tile's K and V^T vectors are already on their way into
//    registers (they are written to LDS after the barrier that ends the tile);
//  * a tile is multiplied by one of two straight-line bodies: one for tiles of which every key is
//    visible to every row of the wave, one that masks (the diagonal, the window's edge, the rows past
//    the sequence's end).  No size is tested inside them, so the compiler can start the LDS reads of a
//    fragment while the products of the one before run;
//  * the rows of a 16-key score tile are assigned to keys so that a lane's eight probabilities of a
//    32-key step belong to eight consecutive keys: its V^T fragment is one 16-byte LDS read;
//  * for D <= 128 a wave's 32 rows are ONE tile of v_mfma_f32_32x32x16_bf16, which sustains 2.1 PFLOP/s on
//    gfx950 where the 16x16x32 shape stops near 1.3 (this kernel is bound by the matrix cores); a lane then
//    holds 32 scores of one row, and the row's statistics need one shuffle;
//  * for D <= 128 the LDS holds two tiles, so a tile costs one barrier: the next tile is written to
//    the other half before this one is multiplied.
#include <type_traits>

#include "common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

#define FAST_THREADS 256
#define FAST_BK 64                                         // keys per LDS tile
#define FAST_PAD 8                                         // LDS row padding in elements
#define FAST_TABLE_MAX 4096                                // block-table entries of a sequence kept in LDS

template <int D, int RB, int WAVES>
__global__ void __launch_bounds__(WAVES * QIL_WAVE, WAVES == 4 ? 2 : 1)
attn_tile_bf16_kernel(const bf16_t* __restrict__ q, int q_stride, const bf16_t* __restrict__ k_cache,
                      const bf16_t* __restrict__ v_cache, const int* __restrict__ block_tables, int table_stride,
                      const int* __restrict__ cu_seqlens, const int* __restrict__ seq_starts, bf16_t* __restrict__ out,
                      int heads, int kv_heads, int page_size, int window, float scale, int GH, int chunks, int ps_shift,
                      float* __restrict__ part_acc, float* __restrict__ part_m, float* __restrict__ part_l, int P,
                      int parts) {
  constexpr int FAST_THREADS_ = WAVES * QIL_WAVE;
  constexpr int BK = FAST_BK, QFRAGS = D / 32, DTILES = D / 16, SUB = BK / 16;
  constexpr int K_ROW = D + FAST_PAD, V_ROW = BK + FAST_PAD;
  constexpr int K_ITERS = BK * (D / 8) / FAST_THREADS_, V_ITERS = D * (BK / 8) / FAST_THREADS_;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  constexpr bool TWO = D <= 128;                           // two tiles in LDS
  constexpr int TILE_ELEMS = BK * K_ROW + D * V_ROW;       // K [BK][K_ROW] (rows in score-tile order), then V^T [D][V_ROW]
  bf16_t* tiles = reinterpret_cast<bf16_t*>(lds_raw);
  int* pages = reinterpret_cast<int*>(tiles + (TWO ? 2 : 1) * TILE_ELEMS);   // the block-table entries this block needs

  // Which sequence, row tile and (kv head, head chunk) this block takes.  Blocks go to the 8 XCDs in turn, each
  // with an L2 of its own: when 256 is a multiple of the number of (sequence, kv head, chunk) triples, block id
  // takes triple id % triples, so that an XCD sees the keys and values of few kv heads (one, with one sequence
  // and 8 of them) and its L2 holds them; and of the row tiles, consecutive groups of 256 blocks walk them in
  // opposite directions, so that the two blocks a CU holds make one long and one short pass over the keys.
  int across, seq = blockIdx.y, pair = blockIdx.z;
  const int triples = gridDim.y * gridDim.z, tiles_x = gridDim.x;
  if (QIL_CUS % triples == 0) {
    const int id = blockIdx.x + tiles_x * (blockIdx.y + gridDim.y * blockIdx.z);
    const int triple = id % triples;
    pair = triple % gridDim.z;                          // the XCD (id % 8) goes with the kv head, not with the sequence:
    seq = triple / gridDim.z;                           // a short sequence's idle blocks then fall on all XCDs alike
    // places in spans of 2 * (256 / triples): the first half of a span takes its upper tiles from the top down,
    // the second half its lower tiles from the bottom up (the last span may be shorter)
    const int place = id / triples, span = 2 * (QIL_CUS / triples), base = place / span * span;
    const int size = min(span, tiles_x - base), idx = place - base, upper = (size + 1) / 2;
    across = base + (idx < upper ? size - 1 - idx : idx - upper);
  } else {
    const int linear = tiles_x * (blockIdx.y + gridDim.y * blockIdx.z);
    across = ((linear >> 8) & 1) ? (int)blockIdx.x : tiles_x - 1 - (int)blockIdx.x;
  }
  // parts > 1 (a few row tiles against a long context): grid.z also counts the parts of P keys, and a block
  // leaves float32 partial results (the layout of the split-context row kernels) for the merge kernel
  const int part = pair / (kv_heads * chunks);
  pair -= part * (kv_heads * chunks);
  const int q0 = cu_seqlens[seq], n = cu_seqlens[seq + 1] - q0;
  if (n < 2) return;
  const int RT = WAVES / GH;
  const int block_rows = 16 * RB * RT;
  const int tile_row0 = across * block_rows;
  if (tile_row0 >= n) return;
  const int kvh = pair / chunks, chunk = pair % chunks;
  const int g = heads / kv_heads;
  const int lane = threadIdx.x & (QIL_WAVE - 1), wave = threadIdx.x / QIL_WAVE;
  const int r = lane & 15, kb = lane >> 4;
  const int head_local = chunk * GH + wave % GH, row_group = wave / GH;
  const int wave_row0 = tile_row0 + row_group * 16 * RB;
  const bool wave_active = head_local < g && wave_row0 < n;
  const int head = kvh * g + head_local;
  const int start = seq_starts[seq];

  const int rows_in_block = min(block_rows, n - tile_row0);
  const int pos_first = start + tile_row0;
  int key_end = pos_first + rows_in_block;                             // last position + 1
  int key_begin = window > 0 ? max(0, pos_first - window + 1) : 0;
  if (parts > 1) {                                                     // P is a multiple of the tile's keys
    key_begin = max(key_begin, part * P);
    key_end = min(key_end, (part + 1) * P);
    if (key_begin >= key_end) return;                                  // no row of the block sees a key of this part
  }
  const int first_tile = key_begin / BK * BK;

  // block-table entries of [first_tile, key_end) into LDS
  const int first_page = first_tile >> ps_shift, last_page = (key_end - 1) >> ps_shift;
  {
    const int* table = block_tables + (size_t)seq * table_stride;
    // as the page's place in the cache in units of 256 bytes (a page of one kv head is 1 KB or more; 32 bits reach 1 TB)
    const uint32_t page_units = (uint32_t)kv_heads * page_size * D / 128;
    for (int i = threadIdx.x; i <= last_page - first_page; i += FAST_THREADS_)
      pages[i] = (int)((uint32_t)table[first_page + i] * page_units);
  }

  int my_row[RB], my_pos[RB];
  bool row_valid[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    my_row[b] = wave_row0 + b * 16 + r;
    row_valid[b] = wave_active && my_row[b] < n;
    my_pos[b] = row_valid[b] ? start + my_row[b] : -1;     // a row past the end sees no key
  }
  const int wave_last_pos = start + min(n, wave_row0 + 16 * RB) - 1;   // nothing beyond it is visible to this wave

  // Q fragments: B operands, Q[row r of tile b][dims 32 ks + 8 kb ..]
  bf16x8 qb[RB][QFRAGS];
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    const bf16_t* qrow = q + (size_t)(q0 + (row_valid[b] ? my_row[b] : 0)) * q_stride + (size_t)(wave_active ? head : 0) * D;
#pragma unroll
    for (int ks = 0; ks < QFRAGS; ++ks) {
      uint4 raw = make_uint4(0, 0, 0, 0);
      if (row_valid[b]) raw = *reinterpret_cast<const uint4*>(qrow + ks * 32 + kb * 8);
      qb[b][ks] = __builtin_bit_cast(bf16x8, raw);
    }
  }
  float m[RB], l[RB];
  f32x4 o[RB][DTILES];
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    m[b] = -INFINITY;
    l[b] = 0.f;
#pragma unroll
    for (int t = 0; t < DTILES; ++t) o[b][t] = (f32x4){0.f, 0.f, 0.f, 0.f};
  }

  // WIDE (D <= 128): the wave's 32 rows as one 32 x 32 tile.  Lane = (row lane % 32, half lane / 32):
  //   S^T[key, row] = K Q^T:  A = K rows (LDS), B = Q[row][dims 16 ks + 8 half ..]
  //     -> the lane's 16 scores of a 32-key tile are the keys 16 (j / 2) + 8 half + 4 (j % 2) + e, j, e < 4
  //        (the K rows are placed in LDS accordingly), so that scores 8 s .. 8 s + 7 are the eight
  //        consecutive keys 16 s + 8 half .. of the tile: the B operand of
  //   O^T[dim, row] = V^T P^T:  A = V^T[dim lane % 32][keys 16 s + 8 half ..] (one 16-byte LDS read)
  //     -> the lane holds O[row][dims 32 t + 8 j + 4 half + e].
  constexpr bool WIDE = RB == 2;
  constexpr int WFRAGS = D / 16, WTILES = D / 32;
  const int l32 = lane & 31, half = lane >> 5;
  const int wide_row = wave_row0 + l32;
  const bool wide_valid = wave_active && wide_row < n;
  const int wide_pos = wide_valid ? start + wide_row : -1;
  bf16x8 qw[WFRAGS];
  float wide_m = -INFINITY, wide_l = 0.f;
  f32x16 ow[WTILES];
  if constexpr (WIDE) {
    const bf16_t* qrow = q + (size_t)(q0 + (wide_valid ? wide_row : 0)) * q_stride + (size_t)(wave_active ? head : 0) * D;
#pragma unroll
    for (int ks = 0; ks < WFRAGS; ++ks) {
      uint4 raw = make_uint4(0, 0, 0, 0);
      if (wide_valid) raw = *reinterpret_cast<const uint4*>(qrow + ks * 16 + half * 8);
      qw[ks] = __builtin_bit_cast(bf16x8, raw);
    }
#pragma unroll
    for (int t = 0; t < WTILES; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) ow[t][i] = 0.f;
  }

  // What this thread stages of every tile: K vector it = 16 bytes of key idx / (D / 8), V^T vector it =
  // 8 keys (one 16-byte piece of a page row) of dim idx % D, idx = thread + it * threads.  A wave's 64 vectors of
  // one `it` lie in one page (K: 512 / D consecutive keys, 1 KB in a row; V^T: 64 dims of one group of 8 keys), so
  // the page and everything else that changes from tile to tile is computed once a wave, on the scalar unit, and a
  // lane adds an offset that never changes.  Only the page is kept inside the sequence's needed pages: any place in
  // such a page is memory of the cache, and what lies outside [key_begin, key_end) is zeroed when published.
  // Addresses: 64 bits for the page (a cache may hold more than 2^31 elements), 32 bits within it.
  uint4 k_reg[K_ITERS], v_reg[V_ITERS];
  constexpr int K_WAVE_KEYS = 512 / D, K_IT_KEYS = FAST_THREADS_ * 8 / D;   // keys of a wave's / the block's vectors of one `it`
  constexpr int V_WAVES_PER_GROUP = D / QIL_WAVE;                           // waves that share a group of 8 keys
  static_assert(K_ITERS == V_ITERS, "K and V^T vectors of one `it` cover the same keys");
  const int wave_s = __builtin_amdgcn_readfirstlane(wave);
  const int low_page = key_begin >> ps_shift;
  // The wave's K vectors of `it` are the keys it * K_IT_KEYS + k_wave .. of the tile, its V^T vectors the 8 keys from
  // it * K_IT_KEYS + v_wave on: both in the same page (k_wave / 8 == v_wave / 8, pages hold 8 keys or more).
  const int k_wave = wave_s * K_WAVE_KEYS, v_wave = wave_s / V_WAVES_PER_GROUP * 8;
  const char* k_head = reinterpret_cast<const char*>(k_cache + (size_t)kvh * page_size * D);
  const char* v_head =
      reinterpret_cast<const char*>(v_cache + ((size_t)kvh * D + (wave_s % V_WAVES_PER_GROUP) * QIL_WAVE) * page_size);
  const uint32_t k_lane = lane * 16, v_lane = lane * page_size * 2;          // bytes
  // Lane `it` looks the page of the vectors `it` up, one request ahead: `held` is in a register when it is needed.
  const int held_key = min(lane, K_ITERS - 1) * K_IT_KEYS + k_wave;
  auto look_up = [&](int k0) { return pages[min(max((k0 + held_key) >> ps_shift, low_page), last_page) - first_page]; };
  int held = 0;
  auto request = [&](int k0) {                             // page_size is a power of two here: ps_shift >= 0
    const int in_page = k0 & (page_size - 1);              // 0 unless a page holds more keys than a tile
#pragma unroll
    for (int it = 0; it < K_ITERS; ++it) {
      const size_t page_at = (size_t)(uint32_t)__builtin_amdgcn_readlane(held, it) << 8;
      const uint32_t k_in = (uint32_t)(in_page + ((it * K_IT_KEYS + k_wave) & (page_size - 1))) * (D * 2);
      const uint32_t v_in = (uint32_t)(in_page + ((it * K_IT_KEYS + v_wave) & (page_size - 1))) * 2;
      k_reg[it] = *reinterpret_cast<const uint4*>(k_head + page_at + k_in + k_lane);
      v_reg[it] = *reinterpret_cast<const uint4*>(v_head + page_at + v_in + v_lane);
    }
    held = look_up(k0 + BK);
  };
  // Key kl of a tile (= 32 a + 8 b + 4 c + e) is row 4 b + e of score sub-tile 2 a + c: lane (r, kb) of the
  // score product then holds, in sub-tiles 2 a and 2 a + 1, the keys 32 a + 8 kb .. + 7.  (WIDE: key
  // 32 a + 16 s + 8 h + 4 j + e is row 16 s + 8 j + 4 h + e of 32-key tile a.)
  int k_to[K_ITERS], v_to[V_ITERS];                        // where this thread's vectors go in a tile, in elements
#pragma unroll
  for (int it = 0; it < K_ITERS; ++it) {
    const int idx = threadIdx.x + it * FAST_THREADS_;
    const int kl = idx / (D / 8), dv = (idx % (D / 8)) * 8;
    const int row = WIDE ? (kl >> 5) * 32 + ((kl >> 4) & 1) * 16 + ((kl >> 2) & 1) * 8 + ((kl >> 3) & 1) * 4 + (kl & 3)
                         : ((kl >> 5) * 2 + ((kl >> 2) & 1)) * 16 + ((kl >> 3) & 3) * 4 + (kl & 3);
    k_to[it] = row * K_ROW + dv;
  }
#pragma unroll
  for (int it = 0; it < V_ITERS; ++it) {
    const int idx = threadIdx.x + it * FAST_THREADS_;
    v_to[it] = BK * K_ROW + (idx % D) * V_ROW + (idx / D) * 8;
  }
  auto publish = [&](int k0, bf16_t* tile) {
    if (k0 >= key_begin && k0 + BK <= key_end) {           // no key of the tile needs zeroing
#pragma unroll
      for (int it = 0; it < K_ITERS; ++it) *reinterpret_cast<uint4*>(tile + k_to[it]) = k_reg[it];
#pragma unroll
      for (int it = 0; it < V_ITERS; ++it) *reinterpret_cast<uint4*>(tile + v_to[it]) = v_reg[it];
      return;
    }
#pragma unroll
    for (int it = 0; it < K_ITERS; ++it) {
      const int key = k0 + (threadIdx.x + it * FAST_THREADS_) / (D / 8);
      const bool valid = key >= key_begin && key < key_end;
      *reinterpret_cast<uint4*>(tile + k_to[it]) = valid ? k_reg[it] : make_uint4(0, 0, 0, 0);
    }
#pragma unroll
    for (int it = 0; it < V_ITERS; ++it) {   // zero what lies outside [key_begin, key_end): never written, or someone else's
      const int key = k0 + (threadIdx.x + it * FAST_THREADS_) / D * 8;
      uint32_t w[4] = {v_reg[it].x, v_reg[it].y, v_reg[it].z, v_reg[it].w};
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (!(key + e >= key_begin && key + e < key_end)) w[e >> 1] &= (e & 1) ? 0x0000ffffu : 0xffff0000u;
      *reinterpret_cast<uint4*>(tile + v_to[it]) = make_uint4(w[0], w[1], w[2], w[3]);
    }
  };

  // One tile's arithmetic.  MASKED: keys a row does not see get score -inf (probability 0).
  const float c = scale * 1.44269504088896f;               // p = exp2((s - m) c): the scale enters in the exponent
  auto attend = [&](int k0, const bf16_t* tile, auto masked_tag) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    const bf16_t* Ks = tile;
    const bf16_t* Vt = tile + BK * K_ROW;
    f32x4 s[RB][SUB];
#pragma unroll
    for (int jt = 0; jt < SUB; ++jt) {
      const bf16_t* krow = Ks + (jt * 16 + r) * K_ROW + kb * 8;
#pragma unroll
      for (int b = 0; b < RB; ++b) s[b][jt] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < QFRAGS; ++ks) {
        const bf16x8 a = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(krow + ks * 32));
#pragma unroll
        for (int b = 0; b < RB; ++b) s[b][jt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qb[b][ks], s[b][jt], 0, 0, 0);
      }
    }
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      float mx = -INFINITY;
#pragma unroll
      for (int jt = 0; jt < SUB; ++jt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (MASKED) {
            const int key = k0 + (jt >> 1) * 32 + 8 * kb + (jt & 1) * 4 + i;
            const bool visible = key <= my_pos[b] && (window <= 0 || key > my_pos[b] - window);
            s[b][jt][i] = visible ? s[b][jt][i] : -INFINITY;
          }
          mx = fmaxf(mx, s[b][jt][i]);
        }
      mx = fmaxf(mx, __shfl_xor(mx, 16, QIL_WAVE));
      mx = fmaxf(mx, __shfl_xor(mx, 32, QIL_WAVE));
      const float m_new = fmaxf(m[b], mx);
      const float base = (m_new == -INFINITY) ? 0.f : m_new;                              // exp(-inf - 0) = 0
      const float shift = -base * c;
      const float alpha = (m_new == -INFINITY) ? 1.f : __builtin_amdgcn_exp2f(fmaf(m[b], c, shift));
      float psum = 0.f;
#pragma unroll
      for (int jt = 0; jt < SUB; ++jt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float p = __builtin_amdgcn_exp2f(fmaf(s[b][jt][i], c, shift));
          s[b][jt][i] = p;
          psum += p;
        }
      l[b] = l[b] * alpha + psum;
      if (m_new != m[b]) {                       // nothing to rescale while the maximum stands
#pragma unroll
        for (int t = 0; t < DTILES; ++t)
#pragma unroll
          for (int i = 0; i < 4; ++i) o[b][t][i] *= alpha;
      }
      m[b] = m_new;
    }
#pragma unroll
    for (int st = 0; st < SUB / 2; ++st) {
      bf16x8 pb[RB];
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        uint32_t packed[4];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          packed[i] = pack_bf16(s[b][2 * st][2 * i], s[b][2 * st][2 * i + 1]);
          packed[2 + i] = pack_bf16(s[b][2 * st + 1][2 * i], s[b][2 * st + 1][2 * i + 1]);
        }
        pb[b] = __builtin_bit_cast(bf16x8, make_uint4(packed[0], packed[1], packed[2], packed[3]));
      }
#pragma unroll
      for (int t = 0; t < DTILES; ++t) {
        const bf16x8 a = __builtin_bit_cast(
            bf16x8, *reinterpret_cast<const uint4*>(Vt + (t * 16 + r) * V_ROW + st * 32 + 8 * kb));
#pragma unroll
        for (int b = 0; b < RB; ++b) o[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb[b], o[b][t], 0, 0, 0);
      }
    }
  };

  auto attend_wide = [&](int k0, const bf16_t* tile, auto masked_tag) {
    constexpr bool MASKED = decltype(masked_tag)::value;
    const bf16_t* Ks = tile;
    const bf16_t* Vt = tile + BK * K_ROW;
    f32x16 s[2];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt) {
      const bf16_t* krow = Ks + (kt * 32 + l32) * K_ROW + half * 8;
#pragma unroll
      for (int i = 0; i < 16; ++i) s[kt][i] = 0.f;
#pragma unroll
      for (int ks = 0; ks < WFRAGS; ++ks) {
        const bf16x8 a = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4*>(krow + ks * 16));
        s[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, qw[ks], s[kt], 0, 0, 0);
      }
    }
    float mx = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        if (MASKED) {
          const int key = k0 + 32 * kt + 16 * (i >> 3) + 8 * half + (i & 7);      // j = i / 4, e = i % 4
          const bool visible = key <= wide_pos && (window <= 0 || key > wide_pos - window);
          s[kt][i] = visible ? s[kt][i] : -INFINITY;
        }
        mx = fmaxf(mx, s[kt][i]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 32, QIL_WAVE));
    const float m_new = fmaxf(wide_m, mx);
    const float base = (m_new == -INFINITY) ? 0.f : m_new;                              // exp(-inf - 0) = 0
    const float shift = -base * c;
    const float alpha = (m_new == -INFINITY) ? 1.f : __builtin_amdgcn_exp2f(fmaf(wide_m, c, shift));
    float psum = 0.f;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float p = __builtin_amdgcn_exp2f(fmaf(s[kt][i], c, shift));
        s[kt][i] = p;
        psum += p;
      }
    wide_l = wide_l * alpha + psum;
    if (m_new != wide_m) {                       // nothing to rescale while the maximum stands
#pragma unroll
      for (int t = 0; t < WTILES; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) ow[t][i] *= alpha;
    }
    wide_m = m_new;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        const bf16x8 pb = __builtin_bit_cast(
            bf16x8, make_uint4(pack_bf16(s[kt][8 * st], s[kt][8 * st + 1]), pack_bf16(s[kt][8 * st + 2], s[kt][8 * st + 3]),
                               pack_bf16(s[kt][8 * st + 4], s[kt][8 * st + 5]), pack_bf16(s[kt][8 * st + 6], s[kt][8 * st + 7])));
#pragma unroll
        for (int t = 0; t < WTILES; ++t) {
          const bf16x8 a = __builtin_bit_cast(
              bf16x8, *reinterpret_cast<const uint4*>(Vt + (t * 32 + l32) * V_ROW + 32 * kt + 16 * st + 8 * half));
          ow[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, pb, ow[t], 0, 0, 0);
        }
      }
  };
  auto attend_tile = [&](int k0, const bf16_t* tile) {
    if (wave_active && k0 <= wave_last_pos) {
      // (rows past the end hold zeros for queries and are not stored: they may see anything)
      const bool all_visible = k0 + BK - 1 <= start + wave_row0 &&
                               (window <= 0 || k0 > wave_last_pos - window);
      if constexpr (WIDE) {
        if (all_visible) attend_wide(k0, tile, std::false_type());
        else attend_wide(k0, tile, std::true_type());
      } else {
        if (all_visible) attend(k0, tile, std::false_type());
        else attend(k0, tile, std::true_type());
      }
    }
  };
  __syncthreads();                                         // the table entries are in place
  held = look_up(first_tile);
  request(first_tile);
  if (TWO) {
    publish(first_tile, tiles);
    if (first_tile + BK < key_end) request(first_tile + BK);
    __syncthreads();
    int half = 0;
    for (int k0 = first_tile; k0 < key_end; k0 += BK, half ^= 1) {
      // the registers hold the next tile; the other half of the LDS was last read before the barrier
      if (k0 + BK < key_end) {
        publish(k0 + BK, tiles + (half ^ 1) * TILE_ELEMS);
        if (k0 + 2 * BK < key_end) request(k0 + 2 * BK);
      }
      attend_tile(k0, tiles + half * TILE_ELEMS);
      __syncthreads();
    }
  } else {
    for (int k0 = first_tile; k0 < key_end; k0 += BK) {
      __syncthreads();                                     // the previous tile is consumed
      publish(k0, tiles);
      __syncthreads();
      if (k0 + BK < key_end) request(k0 + BK);
      attend_tile(k0, tiles);
    }
  }

  if (!wave_active) return;
  if constexpr (WIDE) {
    const float total = wide_l + __shfl_xor(wide_l, 32, QIL_WAVE);
    if (!wide_valid) return;
    if (parts > 1) {
      // acc [row, head, part, d] unnormalised, m (the maximum in the exponent's units) and l [row, head, part]; a row
      // that sees no key of this part leaves m = -inf, l = 0 in a cell the merge does not read
      const size_t cell = ((size_t)(q0 + wide_row) * heads + head) * parts + part;
#pragma unroll
      for (int t = 0; t < WTILES; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          *reinterpret_cast<float4*>(part_acc + cell * D + 32 * t + 8 * j + 4 * half) =
              make_float4(ow[t][4 * j], ow[t][4 * j + 1], ow[t][4 * j + 2], ow[t][4 * j + 3]);
      if (half == 0) {
        part_m[cell] = wide_m == -INFINITY ? -INFINITY : wide_m * scale;
        part_l[cell] = total;
      }
      return;
    }
    const float inv = 1.f / total;
    bf16_t* orow = out + ((size_t)(q0 + wide_row) * heads + head) * D;
#pragma unroll
    for (int t = 0; t < WTILES; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j)                           // dims 32 t + 8 j + 4 half + e, e < 4: 8 bytes
        *reinterpret_cast<uint2*>(orow + 32 * t + 8 * j + 4 * half) =
            make_uint2(pack_bf16(ow[t][4 * j] * inv, ow[t][4 * j + 1] * inv), pack_bf16(ow[t][4 * j + 2] * inv, ow[t][4 * j + 3] * inv));
    return;
  }
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    float total = l[b];
    total += __shfl_xor(total, 16, QIL_WAVE);
    total += __shfl_xor(total, 32, QIL_WAVE);
    if (!row_valid[b]) continue;
    const float inv = 1.f / total;
    bf16_t* orow = out + ((size_t)(q0 + my_row[b]) * heads + head) * D;
#pragma unroll
    for (int t = 0; t < DTILES; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) st(orow + t * 16 + 4 * kb + i, o[b][t][i] * inv);
  }
}

template <int D, int RB, int WAVES>
static int launch_fast(const void* q, int q_stride, const void* k_cache, const void* v_cache, const int* block_tables,
                       int table_stride, const int* cu_seqlens, const int* seq_starts, void* out, int n_seqs,
                       int max_query, int heads, int kv_heads, int page_size, int window, float scale, hipStream_t s,
                       float* workspace = nullptr, int total_rows = 0, int P = 0, int parts = 1) {
  const int g = heads / kv_heads;
  const int GH = g >= 3 ? 4 : g, chunks = (g + GH - 1) / GH, RT = WAVES / GH;
  const size_t lds = (D <= 128 ? 2 : 1) * ((size_t)FAST_BK * (D + FAST_PAD) + (size_t)D * (FAST_BK + FAST_PAD)) * sizeof(bf16_t) +
                     (size_t)table_stride * sizeof(int);
  auto kernel = attn_tile_bf16_kernel<D, RB, WAVES>;
  static size_t granted = 0;                     // per instantiation
  if (lds > 64 * 1024 && lds > granted) {
    hipError_t e = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return (int)e;
    granted = lds;
  }
  dim3 grid((max_query + 16 * RB * RT - 1) / (16 * RB * RT), n_seqs, kv_heads * chunks * parts);
  float* part_m = workspace ? workspace + (size_t)total_rows * heads * parts * D : nullptr;
  float* part_l = part_m ? part_m + (size_t)total_rows * heads * parts : nullptr;
  int ps_shift = -1;                                      // log2 of a power-of-two page size
  for (int b = 0; b < 30; ++b)
    if (page_size == (1 << b)) ps_shift = b;
  hipLaunchKernelGGL(kernel, grid, dim3(WAVES * QIL_WAVE), lds, s, (const bf16_t*)q, q_stride, (const bf16_t*)k_cache,
                     (const bf16_t*)v_cache, block_tables, table_stride, cu_seqlens, seq_starts, (bf16_t*)out, heads,
                     kv_heads, page_size, window, scale, GH, chunks, ps_shift, workspace, part_m, part_l, P, parts);
  return (int)hipGetLastError();
}

// The kernel for head size 128 (attention_prompt.hip).
extern "C" int qil_attn_prompt(const void* q, int q_stride, const void* k_cache, const void* v_cache,
                               const int* block_tables, int table_stride, const int* cu_seqlens, const int* seq_starts,
                               void* out, int n_seqs, int max_query, int heads, int kv_heads, int page_size, int window,
                               float scale, int waves, void* workspace, int total_rows, int P, int parts, hipStream_t s);

static int tile_waves_override = 0;                       // tuning runs and tests: 4 or 16 forces the block shape
extern "C" void qil_attn_tile_waves(int waves) { tile_waves_override = waves; }

// 1 if the kernel of this file takes the sizes (bfloat16 only).
extern "C" int qil_attn_tile_bf16_takes(int d, int page_size, int table_stride) {
  return (d == 64 || d == 128 || d == 256) && page_size >= 8 && (page_size & (page_size - 1)) == 0 &&
         table_stride >= 1 && table_stride <= FAST_TABLE_MAX;
}

// Waves a block of the head-128 kernel: 4, or 16 for 8 waves in two groups that split a block's keys, so that every SIMD has two waves.
// The groups pay where blocks of 4 waves are fewer than CUs, or few more, and a block passes ten tiles of keys or more (``keys``: of the
// longest sequence, as far as the host knows); with many more blocks the SIMDs are full anyway and the merge at the end only costs, as it
// does where the tiles are few.  us in 4 waves / 8, whole prompts, 16 heads in 8 groups: 100 tokens 8.2 / 9.6, 301 11.7 / 12.7, 577
// 16.5 / 16.3, 600 16.8 / 16.4, 700 18.5 / 18.2, 1,000 23.3 / 21.3, 2,000 40.7 / 34.6, 2,560 (320 blocks) 51.8 / 42.8, 2,900 (368)
// 58.5 / 57.7; two of 1,300 (336) 31.1 / 34.0; 32 heads: 900 (232) 22.3 / 21.1, 1,280 (320) 30.6 / 29.0, 1,400 (352) 32.6 / 36.3, 2,048 48.5 / 57.5;
// two of 600 (304) 19.7 / 23.6; three of 301 and 16 heads 12.0 / 13.0.
// Portions behind a history, 16 / 32 heads: 64 rows behind 400 keys 15.4 / 16.3 and 16.2 / 16.3, 128 behind 500 18.0 / 17.6 and 18.4 / 17.9,
// 256 behind 500 20.2 / 19.3 and 20.6 / 19.7, 33 behind 700 19.4 / 18.1 and 20.3 / 19.4, 64 behind 900 23.6 / 22.6 and 24.5 / 22.7; beside rows
// alone (their kernel included) 64 behind 700 and a row of 800 29.0 / 28.1, 64 behind 300 and one of 900 23.2 / 23.7, two of 300 behind 600 and
// one of 950 32.1 / 31.3.
// From 1,024 keys on fewer blocks than CUs have their keys cut into parts before they come here (qil_attn_tile_parts), so that the groups
// get as many blocks as CUs and up to 64 more: 32 heads, four of 256 behind 1,500 40.6 / 37.7, eight of 128 behind 1,000 29.4 / 28.5.
extern "C" int qil_attn_prompt_waves(int n_seqs, int max_query, int keys, int heads, int kv_heads, int window) {
  const int g = heads / kv_heads, gh = g >= 3 ? 4 : g, rows = 32 * (4 / gh);
  const long blocks = (long)((max_query + rows - 1) / rows) * n_seqs * kv_heads * ((g + gh - 1) / gh);
  if (window > 0 || keys <= 9 * FAST_BK) return 4;
  return blocks <= (max_query >= 1024 ? QIL_CUS + 64 : QIL_CUS) ? 16 : 4;
}

// The arguments of qil_attn_tile (attention_tile.hip), which calls this when the sizes are taken.  keys: of the longest
// sequence of several rows, where the host knows it, else the most rows of one.
extern "C" int qil_attn_tile_bf16(const void* q, int q_stride, const void* k_cache, const void* v_cache,
                                  const int* block_tables, int table_stride, const int* cu_seqlens,
                                  const int* seq_starts, void* out, int n_seqs, int max_query, int keys, int heads,
                                  int kv_heads, int d, int page_size, int window, float scale, hipStream_t s) {
  if (n_seqs == 0 || max_query < 2) return 0;
  if (!qil_attn_tile_bf16_takes(d, page_size, table_stride) || heads % kv_heads || n_seqs > 65535 ||
      kv_heads * 2 > 65535)
    return -1;
  if (d == 64)
    return launch_fast<64, 2, 4>(q, q_stride, k_cache, v_cache, block_tables, table_stride, cu_seqlens, seq_starts, out,
                                 n_seqs, max_query, heads, kv_heads, page_size, window, scale, s);
  // Head size 128 has a kernel of its own (attention_prompt.hip), in blocks of 4 waves (32 rows of 4 heads).
  if (d == 128) {
    // (Blocks of 8 waves that share a staged tile of keys, 64 rows of 4 heads, were 8 % faster from 8,192 tokens on
    // and are not used: with 64 query heads in 8 groups, two chunks of heads a group, a 2,048-row sequence beside a
    // 64-row one gave, about once in 2,000 calls inside a model, results that differed from one run to the next in a
    // few rows by the rounding of a bfloat16; with 4 waves, or without the placement of blocks by XCD, never in as
    // many calls; nor with the model's large products on this library's own kernels instead of the GPU BLAS, so the
    // difference is probably made in a BLAS product under that timing.  The shape gains nothing any more and stays out.)
    int waves = qil_attn_prompt_waves(n_seqs, max_query, keys, heads, kv_heads, window);
    if (tile_waves_override) waves = tile_waves_override;   // 4 or 16 (the two groups)
    if (waves == 16 && window > 0) waves = 4;
    return qil_attn_prompt(q, q_stride, k_cache, v_cache, block_tables, table_stride, cu_seqlens, seq_starts, out, n_seqs,
                           max_query, heads, kv_heads, page_size, window, scale, waves, nullptr, 0, 0, 1, s);
  }
  return launch_fast<256, 1, 4>(q, q_stride, k_cache, v_cache, block_tables, table_stride, cu_seqlens, seq_starts, out,
                                n_seqs, max_query, heads, kv_heads, page_size, window, scale, s);
}

// Keys in parts: a portion of a prompt deep in a long context is a few row tiles, each with thousands of keys ahead of
// it, and fewer blocks than the chip has CUs.  Returns the number of parts to cut the keys into (1: do not) and
// their size in *P: about two blocks a CU, parts of at least 256 keys, at most 16 of them.
extern "C" int qil_attn_tile_parts(int n_seqs, int max_query, int heads, int kv_heads, int d, int page_size,
                                   int table_stride, int max_context, int* P) {
  *P = 0;
  if ((d != 64 && d != 128) || !qil_attn_tile_bf16_takes(d, page_size, table_stride) || heads % kv_heads ||
      max_query < 2 || max_context < 1024)
    return 1;
  const int g = heads / kv_heads, gh = g >= 3 ? 4 : g, rows = 32 * (4 / gh);
  const long blocks = (long)((max_query + rows - 1) / rows) * n_seqs * kv_heads * ((g + gh - 1) / gh);
  if (blocks >= QIL_CUS) return 1;
  const int want = (int)min(16L, (2 * QIL_CUS + blocks - 1) / blocks);
  int part = ((max_context + want - 1) / want + FAST_BK - 1) / FAST_BK * FAST_BK;
  part = max(part, 256);
  const int parts = (max_context + part - 1) / part;
  if (parts < 2) return 1;
  *P = part;
  return parts;
}

// qil_attn_tile_bf16 with the keys in `parts` parts of P keys (P a multiple of 64, head size 64 or 128): every row
// of a sequence of two or more rows gets float32 partial results in `workspace` (qil_attn_rows_workspace bytes for
// all `total_rows` rows of the step, indexed by the step's row), which qil_attn_merge then turns into `out`.  The
// cells of rows that are alone in their sequence stay unwritten.
extern "C" int qil_attn_tile_bf16_parts(const void* q, int q_stride, const void* k_cache, const void* v_cache,
                                        const int* block_tables, int table_stride, const int* cu_seqlens,
                                        const int* seq_starts, void* workspace, int total_rows, int n_seqs,
                                        int max_query, int heads, int kv_heads, int d, int page_size, int window,
                                        float scale, int P, int parts, hipStream_t s) {
  if (n_seqs == 0 || max_query < 2) return 0;
  if ((d != 64 && d != 128) || !qil_attn_tile_bf16_takes(d, page_size, table_stride) || heads % kv_heads ||
      n_seqs > 65535 || parts < 2 || P < FAST_BK || P % FAST_BK || !workspace || total_rows < 1 ||
      (long)kv_heads * 2 * parts > 65535)
    return -1;
  if (d == 64)
    return launch_fast<64, 2, 4>(q, q_stride, k_cache, v_cache, block_tables, table_stride, cu_seqlens, seq_starts,
                                 nullptr, n_seqs, max_query, heads, kv_heads, page_size, window, scale, s,
                                 (float*)workspace, total_rows, P, parts);
  return qil_attn_prompt(q, q_stride, k_cache, v_cache, block_tables, table_stride, cu_seqlens, seq_starts, nullptr,
                         n_seqs, max_query, heads, kv_heads, page_size, window, scale, 4, workspace, total_rows, P, parts,
                         s);
}
