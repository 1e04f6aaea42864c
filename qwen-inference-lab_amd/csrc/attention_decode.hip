// Split-context attention of single rows (decoded tokens) on the matrix cores, bfloat16.
//
// Same task and the same partial results as the row kernel in attention_rows.hip (a block owns
// the keys [part * P, (part + 1) * P) of one row and one kv head and serves the whole group of
// query heads reading that kv head; the merge kernel there combines the parts), but the operands
// go from global memory straight into v_mfma_f32_16x16x32_bf16, with no staging in LDS:
//
//   S^T[key, head] = sum_dim K[key, dim] Q[head, dim]     A = K rows      (K is [.., page_size, d])
//   O^T[dim, head] = sum_key V^T[dim, key] P^T[key, head] A = V^T rows    (V is [.., d, page_size])
//
// The 16 columns of a tile are the g query heads of the kv head (columns from g on are zero), so
// a lane holds the scores of ONE head for eight keys (8 (lane / 16) + j of a 32-key step: the rows
// of the two 16-key score tiles are assigned to keys accordingly), and softmax statistics are
// per-lane scalars reduced over the 4 lane groups by two shuffles (qil/paged_attention.py:27-41
// computes the same maxima, sums and weighted values in float32).  Each of the block's waves
// takes every waves-th 32-key step and keeps its own running (m, l, O); they meet in LDS once.
//
// Invisible keys (j > position, or outside the window) may lie in pages that were never
// written or belong to someone else: their scores are replaced, not multiplied, and their V
// elements are zeroed before the product, so garbage (even NaN) cannot enter a sum.
//
// keep > 0: the first `keep` keys stay visible behind a window; steps and parts then count places (key_span.h).
// slopes: slopes[h] * (position - key) is taken off head h's scaled score.
//
// Takes page_size % 8 == 0, d % 16 == 0, d <= 256, g <= 16; other sizes go to the row kernel.
#include <algorithm>

#include "common.h"
#include "fused_qkv.h"
#include "key_span.h"
#include "qk_math.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

#define PLAN_MOST_ROWS 128                                 // rows a plan may share the blocks out to
#define DEC_MAX_WAVES 8                                    // waves of a block; each takes every waves-th 32-key step

// Keys and values are read once a step by one block (the whole group of query heads is served by it).
__device__ __forceinline__ uint4 once4(const bf16_t* p) {
  const qil_u32x4 v = load_once(p);
  return make_uint4(v[0], v[1], v[2], v[3]);
}
__device__ __forceinline__ uint4 pack8(const float* v) {
  return make_uint4(pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7]));
}

// What the first loads need stands in the first 56 bytes of the arguments, which arrive in registers; the rest and the row's
// position and sequence are asked for in batches (a dozen reads of arguments, each waited for by itself, and 10 KB of sines to fetch
// past stood before the first load of data: 8 rows of 2,000 keys 18.8 -> 17.9 us).
// FUSED: fused_qkv.h; FREQUENCIES: its rotation is made from frequencies, not read from tables; ANY_PAGE: pages whose size is no power of
// two.  WHOLE: d == DMAX (always so when FUSED).  PAIRS (not FUSED): a wave has the keys and values of two of its steps in flight.
template <int DMAX, bool FUSED, bool WHOLE = FUSED, bool PAIRS = false, bool FREQUENCIES = false, bool ANY_PAGE = !FUSED>
__global__ void __launch_bounds__(DEC_MAX_WAVES * QIL_WAVE)
attn_decode_kernel(const int* __restrict__ plan, const int* __restrict__ positions, const int* __restrict__ row_seq,
                   const int* __restrict__ block_tables, const bf16_t* __restrict__ k_cache, const bf16_t* __restrict__ v_cache,
                   int table_stride, int P, int heads, int kv_heads, int page_size, int window, int keep, int d, int parts,
                   float scale, float softcap, const int* __restrict__ row_index, const float* __restrict__ sinks,
                   const float* __restrict__ slopes, const bf16_t* __restrict__ q, int q_stride, float* __restrict__ part_acc,
                   float* __restrict__ part_m, float* __restrict__ part_l, bf16_t* __restrict__ out, int* __restrict__ part_keys,
                   FusedQKV fused) {
  constexpr int QFRAGS = DMAX / 32, DTILES = DMAX / 16;
  constexpr int TG = DMAX / 8, HPP = QIL_WAVE / TG;          // lanes of a head (8 elements each), heads a wave
  if (WHOLE) d = DMAX;                                      // what the host has checked, known to the compiler: no
                                                            // condition on the head size stays in the loops
  extern __shared__ float lds[];
  int slot_row = blockIdx.x, part = blockIdx.z;
  const int kvh = blockIdx.y;
  if (__builtin_expect(plan != nullptr, 0)) {               // the rows' parts one behind another (attn_plan_kernel)
    const int job = plan[1 + blockIdx.x];
    P = plan[0];
    if (blockIdx.x == 0 && kvh == 0 && threadIdx.x == 0) *part_keys = P;       // for whoever merges the parts
    if (job < 0) return;
    slot_row = job >> 16;
    part = job & 0xffff;
  }
  if constexpr (FUSED) ask_fields(fused);
  const int row = !FUSED && row_index ? row_index[slot_row] : slot_row;
  const int g = heads / kv_heads;
  const int pos = positions[row], sequence = row_seq[row], ctx = pos + 1;
  asm volatile("" ::"s"(pos), "s"(sequence), "s"(slopes));     // one wait for the three
  const KeySpan span(pos, window, keep);
  const int begin = max(part * P, span.first_place()), end = min((part + 1) * P, span.places());      // places
  if (begin >= end) return;
  const int pos_place = pos - span.hole;                   // the row's own key lies behind the hole

  const int lane = threadIdx.x & (QIL_WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / QIL_WAVE), waves = blockDim.x / QIL_WAVE;
  const int r = lane & 15, kb = lane >> 4;
  const int dt = d / 16;
  const int* table = block_tables + (size_t)sequence * table_stride;

  const int first_step = begin / 32;                       // steps of 32 places, numbered from the first place
  const int last_step = (end - 1) / 32;
  const float slope = (slopes && r < g) ? slopes[kvh * g + r] : 0.f;

  // Q fragments: B operand, column r = head kvh * g + r (filled below, after the first loads are on their way)
  bf16x8 qb[QFRAGS];
  // FUSED, behind the cells in which the waves' results meet: the queries [g][TG] chunks, the new key, the new value
  uint4* shared_q = reinterpret_cast<uint4*>(lds + (blockDim.x / QIL_WAVE * g * (d + 2) + 3) / 4 * 4);
  uint4* shared_new = shared_q + g * TG;
  // FUSED: the block whose keys end with the row's own position makes the new key and value, its last wave does that;
  // `owner` is the wave that meets the position among its steps
  const bool new_here = FUSED && fused.writes && pos_place >= begin && pos_place < end;
  const bool owner = new_here && wave == ((pos_place >> 5) - first_step) % waves;

  float m = -INFINITY, l = 0.f;
  f32x4 o[DTILES];
#pragma unroll
  for (int t = 0; t < DTILES; ++t) o[t] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // The page of a key and its place there.  A division by a number that is not known takes forty instructions a lane; a choice at run
  // time is a branch at each of the first loads' addresses (FUSED: by template; with the new key's page no longer waited for ahead of a
  // wave's sums, us a call: 16 heads of 128 in 8 groups, 1 row of 100 keys 7.9 -> 7.4, 8 of 2,048 15.9 -> 14.9; 14 heads of 64 in 2, 1 row of
  // 8,000 7.8 -> 7.2; pages of 24 keys, 4 rows of 300 9.5 -> 8.9).
  const bool shifts = !ANY_PAGE || (!FUSED && (page_size & (page_size - 1)) == 0);
  const int page_shift = __builtin_ctz(page_size);
  auto page_of = [&](int key) __attribute__((always_inline)) { return __builtin_expect(shifts, 1) ? key >> page_shift : key / page_size; };
  auto place_in = [&](int key) __attribute__((always_inline)) { return __builtin_expect(shifts, 1) ? key & (page_size - 1) : key % page_size; };

  // What one 32-key step needs from memory: the K rows of both 16-key sub-tiles and the V^T fragments
  // of every dim tile, found through three entries of the block table.
  struct StepData {
    uint4 k[2][QFRAGS];
    uint4 v[DTILES];                                        // V^T[dim 16 t + r][keys 8 kb .. 8 kb + 7]: 16 bytes of one page row
  };
  auto look_up = [&](int step, int (&page)[3]) __attribute__((always_inline)) {
    const int k0 = span.key(step * 32);
#pragma unroll
    for (int jt = 0; jt < 2; ++jt)
      // row r of sub-tile jt is key 8 (r / 4) + 4 jt + r % 4 of the step, so that a lane's eight
      // scores (rows 4 kb + i of both sub-tiles) are the eight consecutive keys 8 kb .. 8 kb + 7
      page[jt] = table[page_of(min(k0 + 8 * (r >> 2) + 4 * jt + (r & 3), ctx - 1))];   // clamped: an invisible key's score is replaced
    page[2] = table[page_of(min(k0 + 8 * kb, ctx - 1) & ~7)];
  };
  auto request = [&](int step, const int (&page)[3], StepData& data) __attribute__((always_inline)) {
    const int k0 = span.key(step * 32);
#pragma unroll
    for (int jt = 0; jt < 2; ++jt) {
      const int key = min(k0 + 8 * (r >> 2) + 4 * jt + (r & 3), ctx - 1);
      const bf16_t* krow = k_cache + (((size_t)page[jt] * kv_heads + kvh) * page_size + place_in(key)) * (size_t)d;
#pragma unroll
      for (int ks = 0; ks < QFRAGS; ++ks) {
        const int dim = ks * 32 + kb * 8;
        data.k[jt][ks] = (ks * 32 < d && dim < d) ? once4(krow + dim) : make_uint4(0, 0, 0, 0);
      }
    }
    const int key = min(k0 + 8 * kb, ctx - 1) & ~7;
    const bf16_t* vbase = v_cache + ((size_t)page[2] * kv_heads + kvh) * (size_t)d * page_size + place_in(key);
#pragma unroll
    for (int t = 0; t < DTILES; ++t)
      data.v[t] = t < dt ? once4(vbase + (size_t)(t * 16 + r) * page_size) : make_uint4(0, 0, 0, 0);
  };
  auto attend = [&](int step, StepData& data) __attribute__((always_inline)) {
    const int k0 = span.key(step * 32);
    if constexpr (FUSED) {
      if (owner && step == (pos_place >> 5)) {               // the new key and value are not in the pages yet: from LDS
        const int local = pos & 31;                          // key 8 (rr / 4) + 4 jt + rr % 4 of the step
        const int jt_new = (local >> 2) & 1, rr = ((local >> 3) << 2) | (local & 3);
        uint4 piece[QFRAGS];
        uint32_t value[DTILES];
#pragma unroll
        for (int ks = 0; ks < QFRAGS; ++ks) piece[ks] = shared_new[4 * ks + kb];
#pragma unroll
        for (int t = 0; t < DTILES; ++t) value[t] = reinterpret_cast<const bf16_t*>(shared_new + TG)[16 * t + r];
#pragma unroll
        for (int ks = 0; ks < QFRAGS; ++ks)
#pragma unroll
          for (int jt = 0; jt < 2; ++jt)
            if (r == rr && jt == jt_new) data.k[jt][ks] = piece[ks];
        const int j = local & 7;                             // element of the lanes with kb == local / 8
        uint32_t put[4];                                     // the bits of a lane's four words that the new value takes
#pragma unroll
        for (int i = 0; i < 4; ++i) put[i] = kb == (local >> 3) && i == (j >> 1) ? 0xffffu << ((j & 1) * 16) : 0u;
#pragma unroll
        for (int t = 0; t < DTILES; ++t) {
          const uint32_t both = value[t] * 0x10001u;
          data.v[t].x = (data.v[t].x & ~put[0]) | (both & put[0]);
          data.v[t].y = (data.v[t].y & ~put[1]) | (both & put[1]);
          data.v[t].z = (data.v[t].z & ~put[2]) | (both & put[2]);
          data.v[t].w = (data.v[t].w & ~put[3]) | (both & put[3]);
        }
      }
    }
    // ---- scores
    f32x4 s[2];
#pragma unroll
    for (int jt = 0; jt < 2; ++jt) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < QFRAGS; ++ks)
        if (ks * 32 < d) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, data.k[jt][ks]), qb[ks], acc, 0, 0, 0);
      s[jt] = acc;
    }
    float mx = -INFINITY;
    uint32_t seen[2][4];                                    // 0xffff where the key is visible
#pragma unroll
    for (int jt = 0; jt < 2; ++jt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = k0 + 8 * kb + 4 * jt + i;
        const bool visible = span.visible(key);              // (a part ends at a whole step, or where the keys end)
        seen[jt][i] = visible ? 0xffffu : 0u;
        float v = s[jt][i] * scale;
        if (softcap > 0.f) v = soft_cap_fast(v, softcap, 2.88539008177793f / softcap);
        v = fmaf(slope, (float)(key - pos), v);
        if (!visible) v = -INFINITY;
        s[jt][i] = v;
        mx = fmaxf(mx, v);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16, QIL_WAVE));
    mx = fmaxf(mx, __shfl_xor(mx, 32, QIL_WAVE));
    const float m_new = fmaxf(m, mx);
    const float alpha = (m_new == -INFINITY) ? 1.f : __builtin_amdgcn_exp2f((m - m_new) * 1.44269504088896f);
    float psum = 0.f;
#pragma unroll
    for (int jt = 0; jt < 2; ++jt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p = (s[jt][i] == -INFINITY) ? 0.f : __builtin_amdgcn_exp2f((s[jt][i] - m_new) * 1.44269504088896f);
        s[jt][i] = p;
        psum += p;
      }
    l = l * alpha + psum;
    m = m_new;
    // ---- O^T = O^T alpha + V^T P^T
    uint32_t packed[4];
#pragma unroll
    for (int jt = 0; jt < 2; ++jt)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        packed[jt * 2 + i] = pack_bf16(s[jt][2 * i], s[jt][2 * i + 1]);
    const bf16x8 pb = __builtin_bit_cast(bf16x8, make_uint4(packed[0], packed[1], packed[2], packed[3]));
    const uint32_t mask[4] = {seen[0][0] | (seen[0][1] << 16), seen[0][2] | (seen[0][3] << 16),
                              seen[1][0] | (seen[1][1] << 16), seen[1][2] | (seen[1][3] << 16)};
#pragma unroll
    for (int t = 0; t < DTILES; ++t) {
      if (t < dt) {
        const bf16x8 a = __builtin_bit_cast(bf16x8, make_uint4(data.v[t].x & mask[0], data.v[t].y & mask[1],
                                                                data.v[t].z & mask[2], data.v[t].w & mask[3]));
#pragma unroll
        for (int i = 0; i < 4; ++i) o[t][i] *= alpha;
        o[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb, o[t], 0, 0, 0);
      }
    }
  };
  // FUSED: a wave makes HPP of the group's queries, or (the last wave, in its first lane groups) the new key and value.
  // Everything that takes is asked for ahead of the wave's keys and values, behind which it would wait otherwise: a
  // wave's loads come back in order.  What a wave waits for and how many instructions the slowest one has is what binds rows with few
  // keys: with the new key's page looked up first, no load on the way under a condition, the new key and value from LDS (48
  // shuffles before) and the waves' results read at once, a step of 28 layers and one row took 902 -> 888 us, of 12 layers and 8 rows
  // of 2,048 keys 1,352 -> 1,341.  (With the pages looked up a step ahead: one row of 100 keys at 0.6B sizes 1,102 ->
  // 1,068 us a step of 28 layers, eight of 2,000 1,501 -> 1,467; two steps' keys and values in flight a wave do not fit
  // the registers, and blocks of four waves, three a CU, took 30 us where these take 19.)
  const int chunk = lane % TG, sub = lane / TG;
  const bool makes_q = FUSED && wave * HPP < g;            // wave-uniform, as the others
  const bool makes_new = new_here && wave == waves - 1;
  constexpr int AHEAD = 4;                                 // splits of the product whose sums are asked for at once
  float4 sum_lo[AHEAD], sum_hi[AHEAD];
  HeadFactors factors;
  auto column = [&](bool query, int head) __attribute__((always_inline)) { return query ? (kvh * g + min(head, g - 1)) * DMAX + chunk * 8    // past the group: its last head
                                                         : ((sub & 1 ? fused.v_head : heads) + kvh) * DMAX + chunk * 8; };
  auto ask = [&](bool query, int head) __attribute__((always_inline)) {
    const float* from = fused.qkv + (size_t)row * fused.row_elems + column(query, head);
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const float* p = from + (size_t)min(u, fused.splits - 1) * fused.split_stride;
      sum_lo[u] = *reinterpret_cast<const float4*>(p);
      sum_hi[u] = *reinterpret_cast<const float4*>(p + 4);
    }
    // (what a step has no use for is read from where something stands: a load under a condition would make every wait behind it one
    // for all loads, the keys' and values' too)
    const float* weight = query ? fused.q_weight : fused.k_weight;
    load_eight((weight ? weight : fused.qkv) + chunk * 8, factors.w);
    if constexpr (!FREQUENCIES) {
      const bool turns = fused.cos_table && chunk < 2 * (fused.rot >> 4);
      const int half_chunks = fused.rot >> 4, pair = chunk < half_chunks ? chunk : chunk - half_chunks;
      const size_t at = (size_t)pos * (fused.rot >> 1) + pair * 8;
      load_eight(turns ? fused.cos_table + at : fused.qkv, factors.c);
      load_eight(turns ? fused.sin_table + at : fused.qkv, factors.sn);
    } else {
      load_turns<1>(factors, chunk, fused.cos_table, fused.sin_table, pos, fused.rot);
    }
  };
  // A wave's own sums and factors have arrived (the keys and values asked for behind them need not have).
  auto arrived = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) asm volatile("" : "+v"(sum_lo[u].x), "+v"(sum_lo[u].y), "+v"(sum_lo[u].z), "+v"(sum_lo[u].w),
                                                 "+v"(sum_hi[u].x), "+v"(sum_hi[u].y), "+v"(sum_hi[u].z), "+v"(sum_hi[u].w));
#pragma unroll
    for (int e = 0; e < 8; ++e) asm volatile("" : "+v"(factors.w[e]), "+v"(factors.c[e]), "+v"(factors.sn[e]));
  };
  auto answer = [&](bool query, int head, float (&x)[8], float (&plain)[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = 0.f;
    auto add = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
      for (int u = 0; u < AHEAD; ++u)
        if (s0 + u < fused.splits) {
          x[0] += sum_lo[u].x; x[1] += sum_lo[u].y; x[2] += sum_lo[u].z; x[3] += sum_lo[u].w;
          x[4] += sum_hi[u].x; x[5] += sum_hi[u].y; x[6] += sum_hi[u].z; x[7] += sum_hi[u].w;
        }
    };
    add(0);
    for (int s0 = AHEAD; s0 < fused.splits; s0 += AHEAD) {
      const float* from = fused.qkv + (size_t)row * fused.row_elems + column(query, head);
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        const float* p = from + (size_t)min(s0 + u, fused.splits - 1) * fused.split_stride;
        sum_lo[u] = *reinterpret_cast<const float4*>(p);
        sum_hi[u] = *reinterpret_cast<const float4*>(p + 4);
      }
      arrived();
      add(s0);
    }
    add_bias8(x, fused.bias, column(query, head));
#pragma unroll
    for (int e = 0; e < 8; ++e) plain[e] = x[e];
    norm_rope8<bf16_t>(x, chunk, TG, factors, fused.q_weight != nullptr, DMAX, fused.eps, fused.cos_table && fused.rot > 0,
                       fused.rot, fused.rotate_first != 0);
  };
  // The table's entries come first of all: of the wave's first step and of the new key (asked for at its use, behind the keys and values,
  // its wait was one for all of them, before the barrier that everyone's queries stand behind).
  int new_page = 0;
  auto make_queries = [&]() __attribute__((always_inline)) {
    if constexpr (FUSED) {
      auto make = [&](bool query, int base) __attribute__((always_inline)) {
        float x[8], plain[8];
        answer(query, base + sub, x, plain);
        if (query) {
          if (fused.temp_every > 0) {
            const float temperature = query_temperature(pos, fused.temp_coef, fused.temp_every);
  #pragma unroll
            for (int e = 0; e < 8; ++e) x[e] *= temperature;
          }
          if (base + sub < g) shared_q[(base + sub) * TG + chunk] = pack8(x);
        } else {
          const bool value = sub & 1;
          const uint4 made = value ? pack8(plain) : pack8(x);
          if (sub < 2) {                                   // into the pages (qil/cache.py:79-82), and for this row's own step
            shared_new[sub * TG + chunk] = made;
            const size_t page = new_page;
            const int offset = place_in(pos);
            if (!value) {
              bf16_t* k_row = const_cast<bf16_t*>(k_cache) + ((page * kv_heads + kvh) * page_size + offset) * (size_t)DMAX;
              *reinterpret_cast<uint4*>(k_row + chunk * 8) = made;
            } else {
              bf16_t* column = const_cast<bf16_t*>(v_cache) + ((page * kv_heads + kvh) * (size_t)DMAX + chunk * 8) * page_size + offset;
              const uint32_t words[4] = {made.x, made.y, made.z, made.w};
  #pragma unroll
              for (int e = 0; e < 8; ++e) column[(size_t)e * page_size] = (bf16_t)(words[e >> 1] >> ((e & 1) * 16));
            }
          }
        }
      };
      if (makes_q || makes_new) {
        bool query = makes_q;
        int base = wave * HPP;
        make(query, base);
        while (query) {                                      // (once, unless the group is large for the block's waves)
          base += waves * HPP;
          if (base >= g) {
            if (!makes_new) break;
            query = false;
          }
          ask(query, base + sub);
          arrived();                                         // (no load of this rare way may be open where the ways meet)
          make(query, base);
        }
      }
      __syncthreads();
#pragma unroll
      for (int ks = 0; ks < QFRAGS; ++ks)                    // fragment ks of head r = chunk 4 ks + kb of that head
        qb[ks] = __builtin_bit_cast(bf16x8, r < g ? shared_q[r * TG + 4 * ks + kb] : make_uint4(0, 0, 0, 0));
    } else {
#pragma unroll
      for (int ks = 0; ks < QFRAGS; ++ks) {
        const int dim = ks * 32 + kb * 8;
        uint4 raw = make_uint4(0, 0, 0, 0);
        if (r < g && dim < d) raw = *reinterpret_cast<const uint4*>(q + (size_t)row * q_stride + (size_t)(kvh * g + r) * d + dim);
        qb[ks] = __builtin_bit_cast(bf16x8, raw);
      }
    }
  };
  // The loads of a wave's first step go out before its queries are made, so that the two waits overlap, and the table's
  // entries are looked up a step ahead of the loads that need them.
  constexpr bool EARLY = FUSED;
  int step = first_step + wave;
  if constexpr (PAIRS) {
    // both steps' table entries, then both steps' keys and values, then the arithmetic
    int page_a[3], page_b[3];
    StepData a, b;
    auto load_pair = [&]() __attribute__((always_inline)) {
      look_up(step, page_a);
      if (step + waves <= last_step) look_up(step + waves, page_b);
      request(step, page_a, a);
      if (step + waves <= last_step) request(step + waves, page_b, b);
    };
    if (step <= last_step) load_pair();
    make_queries();
    while (step <= last_step) {
      attend(step, a);
      if (step + waves <= last_step) attend(step + waves, b);
      step += 2 * waves;
      if (step <= last_step) load_pair();
    }
  } else {
    int page[3];
    StepData here;
    if constexpr (EARLY) {
      // (every wave looks up and asks: one without a step of its own for the block's last; conditions would cost the waits' counts)
      look_up(min(step, last_step), page);
      if (new_here) new_page = table[page_of(pos)];
      __builtin_amdgcn_sched_barrier(0);
      if (makes_q || makes_new) {
        ask(makes_q, wave * HPP + sub);
        __builtin_amdgcn_sched_barrier(0);
        request(min(step, last_step), page, here);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" : "+v"(new_page));                   // (needed late: held here only so that it is not asked for late)
        arrived();
      } else {
        request(min(step, last_step), page, here);
      }
    } else if (step <= last_step) {
      look_up(step, page);
      request(step, page, here);
    }
    make_queries();
    if (EARLY) look_up(step + waves, page);                  // (clamped: any entry will do where there is no such step)
    if (step <= last_step)
      for (;;) {
        attend(step, here);
        step += waves;
        if (step > last_step) break;
        if (!EARLY) look_up(step, page);
        request(step, page, here);
        if (EARLY) look_up(step + waves, page);
      }
  }

  // ---- the waves' (m, l, O) meet in LDS: [wave][head < g][d + 2]
  l += __shfl_xor(l, 16, QIL_WAVE);
  l += __shfl_xor(l, 32, QIL_WAVE);
  const int cell = d + 2;
  if (r < g) {
    float* mine = lds + ((size_t)wave * g + r) * cell;
    if (kb == 0) { mine[d] = m; mine[d + 1] = l; }
#pragma unroll
    for (int t = 0; t < DTILES; ++t)
      if (t < dt)
#pragma unroll
        for (int i = 0; i < 4; ++i) mine[t * 16 + 4 * kb + i] = o[t][i];
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < g * d; idx += blockDim.x) {
    const int h = idx / d, e = idx - h * d;
    // every wave's cells asked for at once (waves the block does not have: the last one's, not used)
    float mw[DEC_MAX_WAVES], lw[DEC_MAX_WAVES], ow[DEC_MAX_WAVES], mm = -INFINITY;
#pragma unroll
    for (int w = 0; w < DEC_MAX_WAVES; ++w) {
      const float* theirs = lds + ((size_t)min(w, waves - 1) * g + h) * cell;
      mw[w] = theirs[d];
      lw[w] = theirs[d + 1];
      ow[w] = theirs[e];
    }
#pragma unroll
    for (int w = 0; w < DEC_MAX_WAVES; ++w) mm = fmaxf(mm, mw[w]);
    float total = 0.f, ll = 0.f;
#pragma unroll
    for (int w = 0; w < DEC_MAX_WAVES; ++w) {               // fixed order
      const float f = w >= waves || mw[w] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f((mw[w] - mm) * 1.44269504088896f);
      if (w < waves) {
        total += ow[w] * f;
        ll += lw[w] * f;
      }
    }
    const int head = kvh * g + h;
    if (parts == 1) {
      out[((size_t)row * heads + head) * d + e] =
          f32_to_bf16(sinks ? total * sink_reciprocal(ll, mm, sinks[head]) : total / ll);
    } else {
      const size_t c = ((size_t)slot_row * heads + head) * parts + part;
      part_acc[c * d + e] = total;
      if (e == 0) { part_m[c] = mm; part_l[c] = ll; }
    }
  }
}

// How the keys of rows of different lengths are shared out: parts of one size for all rows, the smallest multiple of 32 keys
// (at least `fewest`) that leaves no more than `blocks` parts in all.  plan[0]: the keys of a part; plan[1 + j]: the j-th
// part, row << 16 | part, the rows one behind another, or -1.  One wave, a row a lane and turn; once a step, for all layers.
__global__ void __launch_bounds__(QIL_WAVE)
attn_plan_kernel(const int* __restrict__ positions, const int* __restrict__ row_index, int rows, int blocks, int fewest,
                 int* __restrict__ plan) {
  const int lane = threadIdx.x;
  constexpr int MOST = PLAN_MOST_ROWS / QIL_WAVE;
  int steps[MOST], total = 0;                              // steps of 32 keys
#pragma unroll
  for (int i = 0; i < MOST; ++i) {
    const int r = i * QIL_WAVE + lane;
    steps[i] = r < rows ? (positions[row_index ? row_index[r] : r] + 32) / 32 : 0;
    total += steps[i];
  }
  auto sum = [](int v) {
    for (int o = QIL_WAVE / 2; o > 0; o >>= 1) v += __shfl_xor(v, o, QIL_WAVE);
    return v;
  };
  total = sum(total);
  // parts(L) = sum over the rows of ceil(steps / L) falls with L; at the longest row's length it is the number of rows
  int low = max(fewest / 32, (total + blocks - 1) / blocks), high = max(low, total);
  while (low < high) {
    const int middle = (low + high) / 2;
    int parts = 0;
#pragma unroll
    for (int i = 0; i < MOST; ++i) parts += (steps[i] + middle - 1) / middle;
    if (sum(parts) <= blocks) high = middle;
    else low = middle + 1;
  }
  if (lane == 0) plan[0] = low * 32;
  int at = 0;
  for (int i = 0; i < MOST; ++i) {
    const int parts = (steps[i] + low - 1) / low;
    int before = parts;                                    // the parts of the rows up to this lane's
    for (int o = 1; o < QIL_WAVE; o *= 2) {
      const int other = __shfl_up(before, o, QIL_WAVE);
      if (lane >= o) before += other;
    }
    for (int p = 0; p < parts; ++p) plan[1 + at + before - parts + p] = ((i * QIL_WAVE + lane) << 16) | p;
    at += __shfl(before, QIL_WAVE - 1, QIL_WAVE);
  }
  for (int j = at + lane; j < blocks; j += QIL_WAVE) plan[1 + j] = -1;
}

// plan: int32 [1 + blocks].  rows <= blocks (a part a row fits) and at most PLAN_MOST_ROWS.
extern "C" int qil_attn_plan(const int* positions, const int* row_index, int rows, int blocks, int fewest, int* plan, hipStream_t s) {
  if (rows < 1 || rows > blocks || rows > PLAN_MOST_ROWS || blocks > 32768 || fewest < 32 || fewest % 32) return -1;
  hipLaunchKernelGGL(attn_plan_kernel, dim3(1), dim3(QIL_WAVE), 0, s, positions, row_index, rows, blocks, fewest, plan);
  QIL_RETURN_LAUNCH_STATUS();
}

// A plan counts whole contexts and needs a workspace; the workspace's rows then hold `parts` parts each, as many as the
// longest row can have.
static bool plan_fits(const int* plan, int blocks, int rows, int parts, int window, const void* workspace) {
  return !plan || (blocks >= rows && rows <= PLAN_MOST_ROWS && parts > 1 && window == 0 && workspace);
}

// 1 if the matrix-core decode kernel takes these sizes.
extern "C" int qil_attn_decode_takes(int heads, int kv_heads, int d, int page_size) {
  if (heads % kv_heads || d % 16 || d < 16 || d > 256 || page_size % 8) return 0;
  const int g = heads / kv_heads;
  return g <= 16 && (size_t)DEC_MAX_WAVES * g * (d + 2) * sizeof(float) <= 64 * 1024;
}

// Partial results in the layout of the row kernel (acc [rows, heads, parts, d], then m, then l);
// the caller runs the row kernel's merge when parts > 1.  P must be a multiple of 32; a block has
// `waves` waves (at most 8), best one or two 32-key steps of P for each.  sinks: null, or float32 [heads]:
// exp(sink) joins a head's divisor (here when parts == 1, else in the merge).  slopes: null, or float32 [heads]; keep > 0
// (with a window): the kept first keys, and P and parts count places.  plan: null, or what qil_attn_plan made for these
// rows and `blocks` (no window): blocks take its parts, P is not used, and the keys of a part are left as an int32 behind
// the partial results (four floats more of workspace) for whoever merges them.
extern "C" int qil_attn_decode(const void* q, int q_stride, const void* k_cache, const void* v_cache,
                               const int* block_tables, int table_stride, const int* row_seq, const int* positions,
                               const int* row_index, void* workspace, void* out, int rows, int heads, int kv_heads,
                               int d, int page_size, int window, float scale, int P, int parts, int waves, float softcap, const float* sinks, const float* slopes, int keep,
                               const int* plan, int blocks, hipStream_t s) {
  if (rows == 0) return 0;
  if (!qil_attn_decode_takes(heads, kv_heads, d, page_size) || (!plan && (P % 32 || P < 32)) || parts < 1 || parts > 65535 ||
      kv_heads > 65535 || waves < 1 || waves > DEC_MAX_WAVES || keep < 0 || (keep > 0 && window <= 0) ||
      !plan_fits(plan, blocks, rows, parts, window, workspace))
    return -1;
  const int g = heads / kv_heads;
  float* acc = (float*)workspace;
  float* m = acc ? acc + (size_t)rows * heads * parts * d : nullptr;
  float* l = m ? m + (size_t)rows * heads * parts : nullptr;
  const size_t lds = (size_t)waves * g * (d + 2) * sizeof(float);
  const dim3 grid = plan ? dim3(blocks, kv_heads) : dim3(rows, kv_heads, parts);
  int* part_keys = plan ? reinterpret_cast<int*>(l + (size_t)rows * heads * parts) : nullptr;
  const FusedQKV none = {};
  // Two of a wave's steps in flight (twice the registers) in launches of at most a block a CU: heads of fewer than 128 elements
  // that do not fill their fragments wherever a wave has a second step, heads of 64 from four steps a wave on.  us with one
  // step / with two: 64 rows of 300 keys, 8 heads of 96 in 4, 12.0 / 10.9, 32 rows of 2,000 keys, 8 heads of 32, 26.5 / 23.4,
  // 16 heads of 64 in 8 groups 30.8 / 29.2, but 16 rows of 1,000 keys 12.9 / 13.4; heads of 128 48.6 / 53.
  const bool pairs = (plan ? (long)blocks : (long)rows * parts) * kv_heads <= QIL_CUS && d < 128 &&
                     (plan || (d == 64 ? P >= 128 * waves : P > 32 * waves));
#define QIL_DEC_LAUNCH(DMAX, FUSED, WHOLE, PAIRS, FIELDS, ...)                                                          \
  hipLaunchKernelGGL((attn_decode_kernel<DMAX, FUSED, WHOLE, PAIRS, ##__VA_ARGS__>), grid, dim3(waves * QIL_WAVE), lds, s, plan,   \
                     positions, row_seq, block_tables, (const bf16_t*)k_cache, (const bf16_t*)v_cache, table_stride, P, heads,     \
                     kv_heads, page_size, window, keep, d, parts, scale, softcap, row_index, sinks, slopes, (const bf16_t*)q,     \
                     q_stride, acc, m, l, (bf16_t*)out, part_keys, FIELDS)
  if (d == 64 && pairs) QIL_DEC_LAUNCH(64, false, true, true, none);
  else if (d == 64) QIL_DEC_LAUNCH(64, false, true, false, none);
  else if (d < 64 && pairs) QIL_DEC_LAUNCH(64, false, false, true, none);
  else if (d < 64) QIL_DEC_LAUNCH(64, false, false, false, none);
  else if (d == 128) QIL_DEC_LAUNCH(128, false, true, false, none);
  else if (d < 128 && pairs) QIL_DEC_LAUNCH(128, false, false, true, none);
  else if (d < 128) QIL_DEC_LAUNCH(128, false, false, false, none);
  else if (d == 256) QIL_DEC_LAUNCH(256, false, true, false, none);
  else QIL_DEC_LAUNCH(256, false, false, false, none);
  QIL_RETURN_LAUNCH_STATUS();
}

// 1 if the fused kernel (queries, new key and new value made from the q/k/v product's partial sums) takes
// the sizes: a head of exactly 64 or 128 elements (256 would not fit the registers), a rotated width the
// vector kernel of qk_rope.hip takes.
extern "C" int qil_attn_decode_fused_takes(int heads, int kv_heads, int d, int page_size, int rot) {
  if (!qil_attn_decode_takes(heads, kv_heads, d, page_size) || !(d == 64 || d == 128)) return 0;
  const int half_chunks = rot >> 4;
  return rot == 0 || (rot <= d && rot % 16 == 0 && (half_chunks & (half_chunks - 1)) == 0);
}

// qil_attn_decode with qkv [splits][rows][(heads + 2 kv_heads) d] float32 partial sums in the place of q; the
// rows are the step's rows 0 .. rows-1 (no row index).  q_weight, k_weight: both or neither; cos/sin: both
// [positions][rot / 2], or neither, or a cos_table alone that holds the rot / 2 frequencies (the angles are then made
// in the kernel).  rotate_first: rotate, then norm.  softcap > 0: scores are capped softly after the scale.  writes != 0: the new keys and values go into the caches at the rows'
// positions (the page comes from the block table).  has_kv 0: the rows of qkv hold queries only (a reader; writes must be 0).
// extra_columns: so many more columns follow in every row and are skipped.  bias: null, or float32 by column of q, k and v.
// temp_every > 0: the query temperature of qk_rope.hip.  sinks: null, or float32 [heads] (as in qil_attn_decode).
// shared_kv: the rows hold no values of their own; a value is its key as projected, before norm and rotation.
// slopes, keep: as in qil_attn_decode.
extern "C" int qil_attn_decode_fused(const float* qkv, int splits, const float* q_weight, const float* k_weight,
                                     float eps, const float* cos_table, const float* sin_table, int rot, int writes,
                                     void* k_cache, void* v_cache, const int* block_tables, int table_stride,
                                     const int* row_seq, const int* positions, void* workspace, void* out, int rows,
                                     int heads, int kv_heads, int d, int page_size, int window, float scale, int P,
                                     int parts, int waves, int rotate_first, float softcap,
                                     int has_kv, int extra_columns, const float* bias, float temp_coef, int temp_every,
                                     const float* sinks, int shared_kv, const float* slopes, int keep,
                                     const int* plan, int blocks, hipStream_t s) {
  if (rows == 0) return 0;
  if (keep < 0 || (keep > 0 && window <= 0) || (shared_kv && !has_kv) || !plan_fits(plan, blocks, rows, parts, window, workspace)) return -1;
  if (extra_columns < 0 || temp_every < 0 || (writes && !has_kv) || ((uintptr_t)bias % 16) || extra_columns % 8) return -1;
  if (!qil_attn_decode_fused_takes(heads, kv_heads, d, page_size, cos_table ? rot : 0) || (!plan && (P % 32 || P < 32)) ||
      parts < 1 || parts > 65535 || kv_heads > 65535 || waves < 1 || waves > DEC_MAX_WAVES || splits < 1 ||
      (q_weight == nullptr) != (k_weight == nullptr) || (sin_table != nullptr && cos_table == nullptr) ||
      (((uintptr_t)qkv | (uintptr_t)q_weight | (uintptr_t)k_weight | (uintptr_t)cos_table | (uintptr_t)sin_table |
        (uintptr_t)k_cache) % 16))
    return -1;
  const int g = heads / kv_heads;
  float* acc = (float*)workspace;
  float* m = acc ? acc + (size_t)rows * heads * parts * d : nullptr;
  float* l = m ? m + (size_t)rows * heads * parts : nullptr;
  const size_t lds = ((size_t)waves * g * (d + 2) + 3) / 4 * 4 * sizeof(float) + (size_t)(g + 2) * d * sizeof(bf16_t);
  const dim3 grid = plan ? dim3(blocks, kv_heads) : dim3(rows, kv_heads, parts);
  int* part_keys = plan ? reinterpret_cast<int*>(l + (size_t)rows * heads * parts) : nullptr;
  FusedQKV fused;
  fused.qkv = qkv;
  fused.row_elems = (heads + (has_kv ? (shared_kv ? 1 : 2) * kv_heads : 0)) * d + extra_columns;
  fused.v_head = shared_kv ? heads : heads + kv_heads;
  fused.split_stride = (size_t)rows * fused.row_elems;
  fused.bias = bias; fused.temp_coef = temp_coef; fused.temp_every = temp_every;
  fused.splits = splits;
  fused.q_weight = q_weight; fused.k_weight = k_weight; fused.eps = eps;
  fused.cos_table = cos_table; fused.sin_table = sin_table; fused.rot = cos_table ? rot : 0;
  fused.rotate_first = rotate_first;
  fused.writes = writes;
  const void* q = nullptr;
  const int q_stride = 0;
  const int* row_index = nullptr;
#define QIL_DEC_FUSED(DMAX, FREQUENCIES, ANY_PAGE)                                                                                \
  do {                                                                                                                             \
    static bool granted = false;                           /* per instantiation: more LDS than a kernel has without asking */      \
    if (lds > 64 * 1024 && !granted) {                                                                                             \
      const hipError_t e = hipFuncSetAttribute((const void*)attn_decode_kernel<DMAX, true, true, false, FREQUENCIES, ANY_PAGE>,    \
                                               hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024);                             \
      if (e != hipSuccess) return (int)e;                                                                                          \
      granted = true;                                                                                                              \
    }                                                                                                                              \
    QIL_DEC_LAUNCH(DMAX, true, true, false, fused, FREQUENCIES, ANY_PAGE);                                                         \
  } while (0)
#define QIL_DEC_FUSED_D(FREQUENCIES, ANY_PAGE)                                                                                    \
  do {                                                                                                                             \
    if (d == 64) QIL_DEC_FUSED(64, FREQUENCIES, ANY_PAGE);                                                                         \
    else QIL_DEC_FUSED(128, FREQUENCIES, ANY_PAGE);                                                                                \
  } while (0)
  const bool frequencies = cos_table && !sin_table, any_page = (page_size & (page_size - 1)) != 0;
  if (frequencies) {
    if (any_page) QIL_DEC_FUSED_D(true, true);
    else QIL_DEC_FUSED_D(true, false);
  } else {
    if (any_page) QIL_DEC_FUSED_D(false, true);
    else QIL_DEC_FUSED_D(false, false);
  }
#undef QIL_DEC_FUSED_D
#undef QIL_DEC_FUSED
#undef QIL_DEC_LAUNCH
  QIL_RETURN_LAUNCH_STATUS();
}
