// Split-context attention of single rows (decoded tokens) on the matrix cores, float32: the task, the parts and the partial
// results of attention_decode.hip, with v_mfma_f32_16x16x4_f32, which takes float32 inputs and adds float32 products into
// float32 sums.  Heads of 64 or 128 elements; other sizes go to the row kernel (attention_rows.hip).
//
//   S^T[key, head] = sum_dim K[key, dim] Q[head, dim]     A = K rows      (K is [.., page_size, d])
//   O^T[dim, head] = sum_key V^T[dim, key] P^T[key, head] A = V^T rows    (V is [.., d, page_size])
//
// A product takes four of the index it sums over, one a lane group kb = lane / 16.  That index may be numbered as one likes:
// product i of a piece takes elements (or keys) 4 kb + i, so that a lane's four are neighbours in memory and come as one
// 16-byte load, and a lane's four scores (rows 4 kb + i of a tile) are the probabilities that its four values meet.  A wave's
// step is 16 keys: 8 + 8 loads a lane in flight with heads of 128.
//
// What bounds it: memory where rows are long (64 products of 32 cycles a step of 16 KB: a CU's four matrix cores ask for 32 bytes
// a cycle, 77 B/ns, twice what memory brings a CU); for few short rows the chain position, page, key, score, value and the launch.
// The row kernel walks the keys once for the scores and once for the values with three barriers between, and adds every score
// over 16 lanes on the vector units.  Alone, keys and values from memory, 16 heads in 8 groups, us row kernel / here: 4 rows of 520
// keys 16.8 / 13.0, 8 of 2,048 35.8 / 32.2, 64 of 300 44.4 / 33.7, 33 of 1,000 81.2 / 65.8, 32 heads and 64 rows of 2,048 221.6 /
// 195.4 (5.5 TB/s); 32 heads of 64 in 2 groups, 8 rows of 1,000, 36.2 / 10.9.  (The parts: ops._matrix_part.)
// With the queries, the new key and the new value made inside, a float32 step of 4 rows of 512 keys at 0.6B sizes takes 1,492 us
// instead of 1,662 (12.6 + 5.1 us a layer -> 12.1).
#include <algorithm>

#include "common.h"
#include "fused_qkv.h"
#include "key_span.h"
#include "qk_math.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

#define DEC32_WAVES 4                                      // waves of a block; each takes every fourth step
#define DEC32_STEP 16                                      // keys of a wave's step

__device__ __forceinline__ f32x4 once_f4(const float* p) {
  return __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p));
}

// FUSED: fused_qkv.h; FREQUENCIES: its rotation is made from frequencies, not read from tables.
template <int D, bool FUSED, bool FREQUENCIES = false>
__global__ void __launch_bounds__(DEC32_WAVES * QIL_WAVE)
attn_decode_f32_kernel(const int* __restrict__ positions, const int* __restrict__ row_seq, const int* __restrict__ block_tables,
                       const float* __restrict__ k_cache, const float* __restrict__ v_cache, int table_stride, int P, int heads,
                       int kv_heads, int page_size, int window, int keep, int parts, float scale, float softcap,
                       const int* __restrict__ row_index, const float* __restrict__ sinks, const float* __restrict__ slopes,
                       const float* __restrict__ q, int q_stride, float* __restrict__ part_acc, float* __restrict__ part_m,
                       float* __restrict__ part_l, float* __restrict__ out, FusedQKV fused) {
  constexpr int PIECES = D / 16, TG = D / 8, HPP = QIL_WAVE / TG, CELL = D + 2, waves = DEC32_WAVES;
  extern __shared__ __align__(16) float lds[];
  const int slot_row = blockIdx.x, kvh = blockIdx.y, part = blockIdx.z;
  if constexpr (FUSED) ask_fields(fused);
  const int row = !FUSED && row_index ? row_index[slot_row] : slot_row;
  const int g = heads / kv_heads;
  const int pos = positions[row], sequence = row_seq[row], ctx = pos + 1;
  asm volatile("" ::"s"(pos), "s"(sequence), "s"(slopes));     // one wait for the three
  const KeySpan span(pos, window, keep);
  const int begin = max(part * P, span.first_place()), end = min((part + 1) * P, span.places());      // places
  if (begin >= end) return;
  const int pos_place = pos - span.hole;                   // the row's own key lies behind the hole

  const int lane = threadIdx.x & (QIL_WAVE - 1), wave = threadIdx.x / QIL_WAVE;
  const int r = lane & 15, kb = lane >> 4;
  const int* table = block_tables + (size_t)sequence * table_stride;
  const int first_step = begin / DEC32_STEP, last_step = (end - 1) / DEC32_STEP;
  const float slope = (slopes && r < g) ? slopes[kvh * g + r] : 0.f;

  float* meeting = lds;                                     // [wave][head < g][CELL] the waves' sums, maxima and results
  float* shared_q = lds + waves * g * CELL;                 // FUSED: [g][D]
  float* shared_new = shared_q + g * D;                     // FUSED: the new key, then the new value
  // FUSED: the block whose keys end with the row's own position makes the new key and value, its last wave does that
  const bool new_here = FUSED && fused.writes && pos_place >= begin && pos_place < end;
  const bool owner = new_here && wave == (pos_place / DEC32_STEP - first_step) % waves;

  f32x4 qb[PIECES];                                         // B operand, column r = head kvh * g + r
  float m = -INFINITY, l = 0.f;
  f32x4 o[PIECES];
#pragma unroll
  for (int t = 0; t < PIECES; ++t) o[t] = (f32x4){0.f, 0.f, 0.f, 0.f};

  struct StepData {
    f32x4 k[PIECES];                                        // K[key r][16 c + 4 kb ..]
    f32x4 v[PIECES];                                        // V^T[dim 16 t + r][keys 4 kb ..]
  };
  auto look_up = [&](int step, int (&page)[2]) __attribute__((always_inline)) {
    const int k0 = span.key(step * DEC32_STEP);
    page[0] = table[min(k0 + r, ctx - 1) / page_size];      // clamped: an invisible key's score is replaced
    page[1] = table[(min(k0 + 4 * kb, ctx - 1) & ~3) / page_size];
  };
  auto request = [&](int step, const int (&page)[2], StepData& data) __attribute__((always_inline)) {
    const int k0 = span.key(step * DEC32_STEP);
    const int key = min(k0 + r, ctx - 1), first = min(k0 + 4 * kb, ctx - 1) & ~3;
    const float* krow = k_cache + (((size_t)page[0] * kv_heads + kvh) * page_size + key % page_size) * (size_t)D + 4 * kb;
    const float* vrow = v_cache + (((size_t)page[1] * kv_heads + kvh) * (size_t)D + r) * page_size + first % page_size;
#pragma unroll
    for (int c = 0; c < PIECES; ++c) data.k[c] = once_f4(krow + 16 * c);
#pragma unroll
    for (int t = 0; t < PIECES; ++t) data.v[t] = once_f4(vrow + (size_t)(16 * t) * page_size);
  };
  auto attend = [&](int step, StepData& data) __attribute__((always_inline)) {
    const int k0 = span.key(step * DEC32_STEP);
    if constexpr (FUSED) {
      if (owner && step == pos_place / DEC32_STEP) {         // the new key and value, as they lie in LDS
        const int local = pos % DEC32_STEP, j = local % 4;
#pragma unroll
        for (int c = 0; c < PIECES; ++c) {
          const f32x4 key = *reinterpret_cast<const f32x4*>(&shared_new[16 * c + 4 * kb]);
          const float value = shared_new[D + 16 * c + r];
          if (r == local) data.k[c] = key;
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (kb == local / 4 && i == j) data.v[c][i] = value;
        }
      }
    }
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < PIECES; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) s = __builtin_amdgcn_mfma_f32_16x16x4f32(data.k[c][i], qb[c][i], s, 0, 0, 0);
    float mx = -INFINITY;
    bool seen[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int key = k0 + 4 * kb + i;
      seen[i] = span.visible(key);
      float v = soft_cap(s[i] * scale, softcap);
      if (slopes) v -= slope * (float)(pos - key);
      s[i] = seen[i] ? v : -INFINITY;
      mx = fmaxf(mx, s[i]);
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, QIL_WAVE));
    mx = fmaxf(mx, __shfl_xor(mx, 32, QIL_WAVE));
    const float m_new = fmaxf(m, mx);
    const float alpha = m_new == -INFINITY ? 1.f : expf(m - m_new);
    float sum = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s[i] = s[i] == -INFINITY ? 0.f : expf(s[i] - m_new);
      sum += s[i];
    }
    l = l * alpha + sum;
    m = m_new;
#pragma unroll
    for (int t = 0; t < PIECES; ++t) {
      o[t] *= alpha;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(seen[i] ? data.v[t][i] : 0.f, s[i], o[t], 0, 0, 0);
    }
  };

  // FUSED: a wave makes HPP of the group's queries, or (the last wave, in its first lane groups) the new key and value;
  // everything that takes is asked for ahead of the wave's keys and values, behind which it would wait otherwise.
  const int chunk = lane % TG, sub = lane / TG;
  const bool makes_q = FUSED && wave * HPP < g;             // wave-uniform, as the others
  const bool makes_new = new_here && wave == waves - 1;
  constexpr int AHEAD = 4;                                  // splits of the product whose sums are asked for at once
  float4 sum_lo[AHEAD], sum_hi[AHEAD];
  HeadFactors factors;
  auto column = [&](bool query, int head) __attribute__((always_inline)) {
    return query ? (kvh * g + min(head, g - 1)) * D + chunk * 8                // past the group: its last head
                 : ((sub & 1 ? fused.v_head : heads) + kvh) * D + chunk * 8;
  };
  auto ask_sums = [&](bool query, int head, int s0) __attribute__((always_inline)) {
    const float* from = fused.qkv + (size_t)row * fused.row_elems + column(query, head);
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
      const float* p = from + (size_t)min(s0 + u, fused.splits - 1) * fused.split_stride;
      sum_lo[u] = *reinterpret_cast<const float4*>(p);
      sum_hi[u] = *reinterpret_cast<const float4*>(p + 4);
    }
  };
  auto ask = [&](bool query, int head) __attribute__((always_inline)) {
    ask_sums(query, head, 0);
    const float* weight = query ? fused.q_weight : fused.k_weight;
    if (weight) load_eight(weight + chunk * 8, factors.w);
    if (fused.cos_table && fused.rot > 0) load_turns<FREQUENCIES>(factors, chunk, fused.cos_table, fused.sin_table, pos, fused.rot);
  };
  auto answer = [&](bool query, int head, float (&x)[8], float (&plain)[8]) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = 0.f;
    for (int s0 = 0; s0 < fused.splits; s0 += AHEAD) {
      if (s0) ask_sums(query, head, s0);
#pragma unroll
      for (int u = 0; u < AHEAD; ++u)
        if (s0 + u < fused.splits) {
          x[0] += sum_lo[u].x; x[1] += sum_lo[u].y; x[2] += sum_lo[u].z; x[3] += sum_lo[u].w;
          x[4] += sum_hi[u].x; x[5] += sum_hi[u].y; x[6] += sum_hi[u].z; x[7] += sum_hi[u].w;
        }
    }
    add_bias8(x, fused.bias, column(query, head));
#pragma unroll
    for (int e = 0; e < 8; ++e) plain[e] = x[e];
    norm_rope8<float>(x, chunk, TG, factors, fused.q_weight != nullptr, D, fused.eps, fused.cos_table && fused.rot > 0,
                      fused.rot, fused.rotate_first != 0);
  };
  auto make_queries = [&]() __attribute__((always_inline)) {
    if constexpr (FUSED) {
      if (makes_q || makes_new) {
        bool query = makes_q;
        for (int base = wave * HPP;;) {                      // once, unless the group is large for the block's waves
          float x[8], plain[8];
          answer(query, base + sub, x, plain);
          if (query) {
            if (fused.temp_every > 0) {
              const float temperature = query_temperature(pos, fused.temp_coef, fused.temp_every);
#pragma unroll
              for (int e = 0; e < 8; ++e) x[e] *= temperature;
            }
            if (base + sub < g) store8(&shared_q[(base + sub) * D + chunk * 8], x);
          } else if (sub < 2) {                              // into the pages, and for this row's own step
            const bool value = sub & 1;
            store8(&shared_new[sub * D + chunk * 8], value ? plain : x);
            const size_t at = (size_t)table[pos / page_size] * kv_heads + kvh;
            const int offset = pos % page_size;
            if (!value) {
              store8(const_cast<float*>(k_cache) + (at * page_size + offset) * (size_t)D + chunk * 8, x);
            } else {
              float* column = const_cast<float*>(v_cache) + (at * D + chunk * 8) * page_size + offset;
#pragma unroll
              for (int e = 0; e < 8; ++e) column[(size_t)e * page_size] = plain[e];
            }
          }
          if (!query) break;
          base += waves * HPP;
          if (base >= g) {
            if (!makes_new) break;
            query = false;
          }
          ask(query, base + sub);
        }
      }
      __syncthreads();
#pragma unroll
      for (int c = 0; c < PIECES; ++c)
        qb[c] = r < g ? *reinterpret_cast<const f32x4*>(&shared_q[r * D + 16 * c + 4 * kb]) : (f32x4){0.f, 0.f, 0.f, 0.f};
    } else {
      const float* mine = q + (size_t)row * q_stride + (size_t)(kvh * g + min(r, g - 1)) * D + 4 * kb;
#pragma unroll
      for (int c = 0; c < PIECES; ++c) {
        const f32x4 raw = *reinterpret_cast<const f32x4*>(mine + 16 * c);
        qb[c] = r < g ? raw : (f32x4){0.f, 0.f, 0.f, 0.f};
      }
    }
  };
  if constexpr (FUSED) {
    if (makes_q || makes_new) ask(makes_q, wave * HPP + sub);
  }
  // a wave's first keys and values are asked for before its queries are made; the table's entries a step ahead of the loads
  int step = first_step + wave;
  int page[2];
  StepData here;
  if (step <= last_step) {
    look_up(step, page);
    request(step, page, here);
    look_up(step + waves, page);                             // (clamped: any entry will do where there is no such step)
  }
  make_queries();
  if (step <= last_step)
    for (;;) {
      attend(step, here);
      step += waves;
      if (step > last_step) break;
      request(step, page, here);
      look_up(step + waves, page);
    }

  // ---- the waves' (m, l, O) meet in LDS
  l += __shfl_xor(l, 16, QIL_WAVE);
  l += __shfl_xor(l, 32, QIL_WAVE);
  if (r < g) {
    float* mine = meeting + ((size_t)wave * g + r) * CELL;
    if (kb == 0) { mine[D] = m; mine[D + 1] = l; }
#pragma unroll
    for (int t = 0; t < PIECES; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) mine[t * 16 + 4 * kb + i] = o[t][i];
  }
  __syncthreads();
  for (int idx = threadIdx.x; idx < g * D; idx += blockDim.x) {
    const int h = idx / D, e = idx % D;
    float mm = -INFINITY;
    for (int w = 0; w < waves; ++w) mm = fmaxf(mm, meeting[((size_t)w * g + h) * CELL + D]);
    float total = 0.f, ll = 0.f;
    for (int w = 0; w < waves; ++w) {                        // fixed order
      const float* his = meeting + ((size_t)w * g + h) * CELL;
      const float f = his[D] == -INFINITY ? 0.f : expf(his[D] - mm);
      total += his[e] * f;
      ll += his[D + 1] * f;
    }
    const int head = kvh * g + h;
    if (parts == 1) {
      out[((size_t)row * heads + head) * D + e] = sinks ? total * sink_reciprocal(ll, mm, sinks[head]) : total / ll;
    } else {
      const size_t c = ((size_t)slot_row * heads + head) * parts + part;
      part_acc[c * D + e] = total;
      if (e == 0) { part_m[c] = mm; part_l[c] = ll; }
    }
  }
}

// LDS: the waves' results, and (FUSED) the queries and the new key and value behind them.
static size_t dec32_lds(int g, int d, bool fused) {
  return ((size_t)DEC32_WAVES * g * (d + 2) + (fused ? (size_t)(g + 2) * d : 0)) * sizeof(float);
}

extern "C" {

// 1 if the kernel takes these sizes (fused 1: also with the queries made inside, rot elements rotated).
int qil_attn_decode_f32_takes(int heads, int kv_heads, int d, int page_size, int fused, int rot) {
  if (heads < 1 || kv_heads < 1 || heads % kv_heads || (d != 64 && d != 128) || page_size < 4 || page_size % 4) return 0;
  const int g = heads / kv_heads;
  if (g > 16 || dec32_lds(g, d, fused != 0) > 64 * 1024) return 0;
  const int half_chunks = rot >> 4;
  return !fused || rot == 0 || (rot <= d && rot % 16 == 0 && (half_chunks & (half_chunks - 1)) == 0);
}

// As qil_attn_decode without a plan, float32 throughout; P a multiple of 32 (64 and more keep all waves at work).
int qil_attn_decode_f32(const void* q, int q_stride, const void* k_cache, const void* v_cache, const int* block_tables,
                        int table_stride, const int* row_seq, const int* positions, const int* row_index, void* workspace,
                        void* out, int rows, int heads, int kv_heads, int d, int page_size, int window, float scale, int P,
                        int parts, float softcap, const float* sinks, const float* slopes, int keep, hipStream_t s) {
  if (rows == 0) return 0;
  if (!qil_attn_decode_f32_takes(heads, kv_heads, d, page_size, 0, 0) || P % 32 || P < 32 || parts < 1 || parts > 65535 ||
      kv_heads > 65535 || keep < 0 || (keep > 0 && window <= 0) || (parts > 1 && !workspace) || q_stride % 4 ||
      (((uintptr_t)q | (uintptr_t)k_cache | (uintptr_t)v_cache) % 16))
    return -1;
  const int g = heads / kv_heads;
  float* acc = (float*)workspace;
  float* m = acc ? acc + (size_t)rows * heads * parts * d : nullptr;
  float* l = m ? m + (size_t)rows * heads * parts : nullptr;
  const size_t lds = dec32_lds(g, d, false);
  const dim3 grid(rows, kv_heads, parts);
  const FusedQKV none = {};
#define QIL_DEC32(D, FUSED, FIELDS, ...)                                                                              \
  hipLaunchKernelGGL((attn_decode_f32_kernel<D, FUSED, ##__VA_ARGS__>), grid, dim3(DEC32_WAVES * QIL_WAVE), lds, s, positions, row_seq, \
                     block_tables, (const float*)k_cache, (const float*)v_cache, table_stride, P, heads, kv_heads,      \
                     page_size, window, keep, parts, scale, softcap, row_index, sinks, slopes, (const float*)q, q_stride, \
                     acc, m, l, (float*)out, FIELDS)
  if (d == 64) QIL_DEC32(64, false, none);
  else QIL_DEC32(128, false, none);
  QIL_RETURN_LAUNCH_STATUS();
}

// As qil_attn_decode_fused without a plan, float32 throughout.
int qil_attn_decode_f32_fused(const float* qkv, int splits, const float* q_weight, const float* k_weight, float eps,
                              const float* cos_table, const float* sin_table, int rot, int writes, void* k_cache,
                              void* v_cache, const int* block_tables, int table_stride, const int* row_seq,
                              const int* positions, void* workspace, void* out, int rows, int heads, int kv_heads, int d,
                              int page_size, int window, float scale, int P, int parts, int rotate_first,
                              float softcap, int has_kv, int extra_columns, const float* bias, float temp_coef, int temp_every,
                              const float* sinks, int shared_kv, const float* slopes, int keep, hipStream_t s) {
  if (rows == 0) return 0;
  if (keep < 0 || (keep > 0 && window <= 0) || (shared_kv && !has_kv) || (parts > 1 && !workspace)) return -1;
  if (extra_columns < 0 || temp_every < 0 || (writes && !has_kv) || extra_columns % 8) return -1;
  if (!qil_attn_decode_f32_takes(heads, kv_heads, d, page_size, 1, cos_table ? rot : 0) || P % 32 || P < 32 ||
      parts < 1 || parts > 65535 || kv_heads > 65535 || splits < 1 ||
      (q_weight == nullptr) != (k_weight == nullptr) || (sin_table != nullptr && cos_table == nullptr) ||
      (((uintptr_t)qkv | (uintptr_t)q_weight | (uintptr_t)k_weight | (uintptr_t)cos_table | (uintptr_t)sin_table |
        (uintptr_t)k_cache | (uintptr_t)v_cache | (uintptr_t)bias) % 16))
    return -1;
  const int g = heads / kv_heads;
  float* acc = (float*)workspace;
  float* m = acc ? acc + (size_t)rows * heads * parts * d : nullptr;
  float* l = m ? m + (size_t)rows * heads * parts : nullptr;
  const size_t lds = dec32_lds(g, d, true);
  const dim3 grid(rows, kv_heads, parts);
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
  if (cos_table && !sin_table) {
    if (d == 64) QIL_DEC32(64, true, fused, true);
    else QIL_DEC32(128, true, fused, true);
  } else {
    if (d == 64) QIL_DEC32(64, true, fused);
    else QIL_DEC32(128, true, fused);
  }
#undef QIL_DEC32
  QIL_RETURN_LAUNCH_STATUS();
}

}  // extern "C"
