// The linear recurrences of recurrence.hip (S_t = a_t S_(t-1) + b_t k_t v_t^T, o_t = S_t^T q_t; the same gating modes,
// the same state slot) for long runs of tokens, in blocks of SCAN_BLOCK tokens that are worked on side by side.
//
// With the log gates f_u (keep) and i_s (input) of a block, F_t = f_0 + ... + f_t, e_s = i_s - F_s and the running
// maximum carried into the block m_in (over the state S_in, normaliser n_in that it scales):
//     M_t = max(m_in, e_0 .. e_t)                       m_t = F_t + M_t
//     S_t = exp(m_in - M_t) S_in + sum_(s <= t) exp(e_s - M_t) k_s v_s^T            (every exponent <= 0)
//     o_t = exp(m_in - M_t) S_in^T q_t + sum_(s <= t) exp(e_s - M_t) (q_t . k_s) v_s
// and n_t . q_t the same with 1 for v_s.  With a fixed decay d: exp(e_s - M_t) is d^(t - s) and exp(m_in - M_t) is
// d^(t + 1).  Four kernels, all float32 (sums of gates and their differences in float64, so that the exponent of a
// weight near 1 is not the rounded difference of two large numbers):
//   rotate   queries and keys rotated by position and scaled, once, into float32 rows;
//   sums     per block: U = sum_s w_s k_s v_s^T (and the normaliser's sum_s w_s k_s) with w_s = exp(e_s - max e), what
//            the block adds to the state at its end: a [dim, 64 tokens] x [64 tokens, vdim] product, tiled 64 x 64;
//   carry    block after block, S_out = exp(m_in - M_end) S_in + exp(max e - M_end) U, element by element; every block's
//            S_in replaces its U, the last S_out goes to the state slot;
//   outputs  per block: [q scaled by its carry weight | masked weighted q k^T] x [S_in ; v], tiled 64 tokens x 64 columns.
// The tiled products are float32: on the matrix cores for DECAY and MLSTM at the sizes scan_mfma_takes names, otherwise on
// the vector units (4 x 4 outputs a thread, operands staged in LDS).
//
// QIL_SCAN_CHANNEL (every row i of S decays by a factor of its own, a_t[i] = exp(logsigmoid(z_t[i]) / tau)): with
// G_t[i] the sum of the block's log2 decays of row i up to token t (one more kernel, `decays`, walks them),
//     S_t = diag(2^G_t) S_in + sum_(s <= t) diag(2^(G_t - G_s)) k_s v_s^T
//     o_t = S_in^T (q_t * 2^G_t) + sum_(s <= t) (sum_i q_t[i] k_s[i] 2^(G_t[i] - G_s[i])) v_s
// so `sums` weighs row i of k_s by 2^(G_end[i] - G_s[i]), `carry` keeps row i by 2^G_end[i], and `outputs` makes the
// scores inside the block with the weight inside the sum over i (every exponent <= 0: nothing is divided by a decay).
//
// QIL_SCAN_STEP (a step size d_t per head and token, a_t = exp(rate d_t), b_t = d_t): with F_t the block's sum of rate d,
//     S_t = exp(F_t) S_in + sum_(s <= t) exp(F_t - F_s) d_s k_s v_s^T
// every exponent <= 0 again.  Queries and keys are shared by groups of heads and read where they lie: nothing to rotate.
#include "common.h"
#include "operand.h"

enum { QIL_SCAN_DECAY = 0, QIL_SCAN_MLSTM = 1, QIL_SCAN_CHANNEL = 2, QIL_SCAN_STEP = 3 };
#define SCAN_BLOCK 64
#define SCAN_TOP_TILE 16                                         // recurrence.hip keeps one maximum per 16 state columns

__device__ __forceinline__ float log_sigmoid_c(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }

// Lane t of a wave: F_t and e_t of token t of the block (e = -inf past the block's end).
struct GateLane { double sum, lead; };
__device__ __forceinline__ GateLane gate_lane(const float* __restrict__ gates, const float* __restrict__ gate_bias,
                                              float cap, int row, int h, int heads, bool live, int lane) {
  float in = 0.f, keep = 0.f;
  if (live) {
    in = cap * tanhf((gates[(size_t)row * 2 * heads + h] + gate_bias[h]) / cap);
    keep = log_sigmoid_c(cap * tanhf((gates[(size_t)row * 2 * heads + heads + h] + gate_bias[heads + h]) / cap));
  }
  double sum = keep;
#pragma unroll
  for (int d = 1; d < QIL_WAVE; d <<= 1) {
    const double up = __shfl_up(sum, d, QIL_WAVE);
    if (lane >= d) sum += up;
  }
  GateLane g;
  g.sum = sum;
  g.lead = live ? (double)in - sum : -INFINITY;
  return g;
}

// d^n for n of 0 to 127 by squaring, in float64 (a dozen multiplications, each good to 2^-53: the float32 it is rounded to
// is pow's, which costs a wave 1.5 us).
__device__ __forceinline__ float decay_power(double d, int n) {
  double power = 1.0;
#pragma unroll
  for (int bit = 0; bit < 7; ++bit) {
    if (n >> bit & 1) power *= d;
    d *= d;
  }
  return (float)power;
}

// STEP, lane t: F_t and the step size d_t of token t (0 past the block's end).
struct StepInput { Operand raw; int row, q_off, k_off, groups; };
struct StepLane { double sum; float step; };
__device__ __forceinline__ StepLane step_lane(const StepInput& in, const float* __restrict__ bias, float rate, int row, int h,
                                              bool live, int lane) {
  float step = 0.f;
  if (live) {
    const float v = operand_at(in.raw, (size_t)row * in.row + h) + bias[h];
    step = v > 20.f ? v : log1pf(expf(v));
  }
  double sum = (double)(rate * step);
#pragma unroll
  for (int d = 1; d < QIL_WAVE; d <<= 1) {
    const double up = __shfl_up(sum, d, QIL_WAVE);
    if (lane >= d) sum += up;
  }
  return {sum, step};
}

// Where block c of sequence seq keeps its sums: sequences before it took at most row0 / SCAN_BLOCK + seq places.
__device__ __forceinline__ int block_place(int row0, int seq, int c) { return row0 / SCAN_BLOCK + seq + c; }

// CHANNEL: gsum[row, e] = sum over the block's tokens up to this row of log2(a[e]), e over heads * dim; the sum runs
// in float64 and is rounded once.  grid (blocks of the longest sequence, sequences, heads * dim / 256)
__global__ void __launch_bounds__(256)
scan_decays_kernel(const float* __restrict__ z, float tau, const int* __restrict__ cu_seqlens, float* __restrict__ gsum,
                   int hd) {
  const int c = blockIdx.x, seq = blockIdx.y, e = blockIdx.z * blockDim.x + threadIdx.x;
  const int row0 = cu_seqlens[seq], len = cu_seqlens[seq + 1] - row0;
  if (c * SCAN_BLOCK >= len || e >= hd) return;
  const int r0 = row0 + c * SCAN_BLOCK, lc = min(SCAN_BLOCK, len - c * SCAN_BLOCK);
  double sum = 0.0;
  for (int t0 = 0; t0 < lc; t0 += 8) {
    float in[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) in[u] = z[(size_t)(r0 + min(t0 + u, lc - 1)) * hd + e];
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (t0 + u < lc) {
        sum += (double)(log_sigmoid_c(in[u]) / tau) * 1.4426950408889634;
        gsum[(size_t)(r0 + t0 + u) * hd + e] = (float)sum;
      }
  }
}

// One block a row.  A thread owns one pair of rotated elements (or one that passes through) of a head and meets it in every
// head's query and key, so that its sine and cosine are made once a row and not once an element: 3,044 rows of 2 x 8 heads
// of 128 elements 22.8 -> 12.4 us (37 MB).  blockDim.x is a multiple of the units a head has, dim - rot / 2.
template <typename T>
__global__ void __launch_bounds__(256)
scan_rotate_kernel(const T* __restrict__ proj, int proj_row, int q_off, int k_off, const float* __restrict__ freq, int rot,
                   float q_scale, float k_scale, const int* __restrict__ cu_seqlens, const int* __restrict__ seq_starts,
                   int n_seqs, float* __restrict__ qk, int heads, int dim) {
  const int row = blockIdx.x, half = rot / 2, units = dim - half, hd = heads * dim;
  const int unit = threadIdx.x % units, step = blockDim.x / units;
  const int i = unit < half ? unit : unit + half;
  float sn = 0.f, cs = 1.f;
  if (unit < half) {
    int seq = 0;
    while (seq + 1 < n_seqs && cu_seqlens[seq + 1] <= row) ++seq;
    const float position = (float)(seq_starts[seq] + row - cu_seqlens[seq]);
    sincosf(position * freq[unit], &sn, &cs);
  }
  const T* x = proj + (size_t)row * proj_row;
  float* to = qk + (size_t)row * 2 * hd;
#pragma unroll 4
  for (int place = threadIdx.x / units; place < 2 * heads; place += step) {
    const bool key = place >= heads;
    const int e = (key ? place - heads : place) * dim + i;
    const T* src = x + (key ? k_off : q_off) + e;
    const float scale = key ? k_scale : q_scale, first = ld(src);
    float* out = to + (key ? hd : 0) + e;
    if (unit < half) {
      const float second = ld(src + half);
      out[0] = (first * cs - second * sn) * scale;
      out[half] = (second * cs + first * sn) * scale;
    } else {
      out[0] = first * scale;
    }
  }
}

// Lane s of a wave: what the key and value of token s of block c are worth in the block's sum; the lane of the first token
// of the grid's first z also leaves what the carry needs of the block's gates.
template <int MODE>
__device__ __forceinline__ float sums_weight(const float* __restrict__ gates, const float* __restrict__ gate_bias, float cap,
                                             const float* __restrict__ decay, const float* __restrict__ state,
                                             size_t slot_stride, const int* __restrict__ seq_starts,
                                             const int* __restrict__ seq_slots, double* __restrict__ info,
                                             float* __restrict__ carried, int heads, int dim, int vdim,
                                             const StepInput& steps, int seq, int h, int c, int r0, int lc, size_t at,
                                             bool writes, int lane) {
  const bool live = lane < lc;
  float weight;
  if (MODE == QIL_SCAN_MLSTM) {
    const GateLane g = gate_lane(gates, gate_bias, cap, r0 + (live ? lane : 0), h, heads, live, lane);
    double top = g.lead;
#pragma unroll
    for (int d = QIL_WAVE / 2; d > 0; d >>= 1) top = fmax(top, __shfl_xor(top, d, QIL_WAVE));
    weight = live ? expf((float)(g.lead - top)) : 0.f;
    const double total = __shfl(g.sum, lc - 1, QIL_WAVE);
    if (writes && lane == 0) {
      info[at * 2] = top;
      info[at * 2 + 1] = total;
      if (c == 0) {                                            // the maximum the sequence brings: read before carry writes
        const int tiles = (vdim + SCAN_TOP_TILE - 1) / SCAN_TOP_TILE;
        const float* s_top = state + (size_t)seq_slots[seq] * slot_stride + (size_t)heads * dim * vdim +
                             (size_t)heads * dim + (size_t)h * (tiles + 1);
        carried[at] = seq_starts[seq] == 0 ? 0.f : *s_top;
      }
    }
  } else if (MODE == QIL_SCAN_STEP) {
    const StepLane g = step_lane(steps, gate_bias, decay[h], r0 + (live ? lane : 0), h, live, lane);
    const double total = __shfl(g.sum, lc - 1, QIL_WAVE);
    weight = live ? expf((float)(total - g.sum)) * g.step : 0.f;
    if (writes && lane == 0) info[at * 2] = total;
  } else if (MODE == QIL_SCAN_CHANNEL) {
    weight = live ? 1.f : 0.f;                                 // (the rows' own weights follow below)
  } else {
    weight = live ? decay_power((double)decay[h], lc - 1 - lane) : 0.f;
  }
  return weight;
}

// grid (blocks of the longest sequence, sequences x heads, dim tiles x vdim tiles)
template <typename T, int MODE>
__global__ void __launch_bounds__(256)
scan_sums_kernel(const T* __restrict__ proj, int proj_row, int v_off, const float* __restrict__ qk,
                 const float* __restrict__ gates, const float* __restrict__ gate_bias, float cap,
                 const float* __restrict__ decay, const float* __restrict__ state, size_t slot_stride,
                 const int* __restrict__ cu_seqlens, const int* __restrict__ seq_starts, const int* __restrict__ seq_slots,
                 float* __restrict__ sums, float* __restrict__ norm_sums, double* __restrict__ info,
                 float* __restrict__ carried, int heads, int dim, int vdim, int dim_tiles,
                 const float* __restrict__ gsum, StepInput steps) {
  __shared__ __align__(16) float kw[SCAN_BLOCK][64];
  __shared__ __align__(16) float vs[SCAN_BLOCK][64];
  __shared__ float w[SCAN_BLOCK];
  const int c = blockIdx.x, seq = blockIdx.y / heads, h = blockIdx.y % heads;
  const int it = blockIdx.z % dim_tiles, jt = blockIdx.z / dim_tiles, tid = threadIdx.x;
  const int row0 = cu_seqlens[seq], len = cu_seqlens[seq + 1] - row0;
  if (c * SCAN_BLOCK >= len) return;
  const int r0 = row0 + c * SCAN_BLOCK, lc = min(SCAN_BLOCK, len - c * SCAN_BLOCK);
  const size_t at = (size_t)block_place(row0, seq, c) * heads + h;
  if (tid < QIL_WAVE)
    w[tid] = sums_weight<MODE>(gates, gate_bias, cap, decay, state, slot_stride, seq_starts, seq_slots, info, carried, heads,
                               dim, vdim, steps, seq, h, c, r0, lc, at, blockIdx.z == 0, tid);
  __syncthreads();
  const size_t hd = (size_t)heads * dim;
  const int group = MODE == QIL_SCAN_STEP ? h / (heads / steps.groups) : h;
  for (int idx = tid; idx < SCAN_BLOCK * 64; idx += 256) {
    const int s = idx / 64, x = idx % 64, i = it * 64 + x, j = jt * 64 + x;
    float weight = w[s];
    if (MODE == QIL_SCAN_CHANNEL && s < lc && i < dim)
      weight = __builtin_amdgcn_exp2f(gsum[(size_t)(r0 + lc - 1) * hd + (size_t)h * dim + i] -
                                      gsum[(size_t)(r0 + s) * hd + (size_t)h * dim + i]);
    if (MODE == QIL_SCAN_STEP)
      kw[s][x] = (s < lc && i < dim) ? weight * ld(proj + (size_t)(r0 + s) * proj_row + steps.k_off + group * dim + i) : 0.f;
    else
      kw[s][x] = (s < lc && i < dim) ? weight * qk[(size_t)(r0 + s) * 2 * hd + hd + (size_t)h * dim + i] : 0.f;
    vs[s][x] = (s < lc && j < vdim) ? ld(proj + (size_t)(r0 + s) * proj_row + v_off + h * vdim + j) : 0.f;
  }
  __syncthreads();
  const int ti = tid / 16, tj = tid % 16;
  float acc[4][4] = {};
  for (int s = 0; s < lc; ++s) {
    const float4 a4 = *reinterpret_cast<const float4*>(&kw[s][ti * 4]);
    const float4 b4 = *reinterpret_cast<const float4*>(&vs[s][tj * 4]);
    const float a[4] = {a4.x, a4.y, a4.z, a4.w}, b[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[r][q] += a[r] * b[q];
  }
  float* u = sums + at * dim * vdim;
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int i = it * 64 + ti * 4 + r, j = jt * 64 + tj * 4 + q;
      if (i < dim && j < vdim) u[(size_t)i * vdim + j] = acc[r][q];
    }
  if (MODE == QIL_SCAN_MLSTM && jt == 0 && tid < 64 && it * 64 + tid < dim) {
    float total = 0.f;
    for (int s = 0; s < lc; ++s) total += kw[s][tid];
    norm_sums[at * dim + it * 64 + tid] = total;
  }
}

// grid (sequences, heads, elements of a head's state / 256 V): a thread takes V neighbouring elements of S (or of n) block
// after block.  Four where they are aligned and lie in one row of S (V == 4: dim and vdim multiples of 4): 48 blocks of
// 8 heads of 128 x 256 26.8 -> 18.0 us (102 MB).
#define CARRY_AHEAD 8
template <int MODE, int V>
__global__ void __launch_bounds__(256)
scan_carry_kernel(float* __restrict__ sums, float* __restrict__ norm_sums, const double* __restrict__ info,
                  float* __restrict__ carried, const float* __restrict__ decay, float* __restrict__ state,
                  size_t slot_stride, const int* __restrict__ cu_seqlens, const int* __restrict__ seq_starts,
                  const int* __restrict__ seq_slots, int heads, int dim, int vdim, const float* __restrict__ gsum) {
  typedef float Piece __attribute__((ext_vector_type(V)));
  const int seq = blockIdx.x, h = blockIdx.y, e = (blockIdx.z * blockDim.x + threadIdx.x) * V;
  const int mat = dim * vdim, total = mat + (MODE == QIL_SCAN_MLSTM ? dim : 0);
  const int row0 = cu_seqlens[seq], len = cu_seqlens[seq + 1] - row0;
  if (len <= 0 || e >= total) return;
  const bool fresh = seq_starts[seq] == 0;
  const int tiles = (vdim + SCAN_TOP_TILE - 1) / SCAN_TOP_TILE;
  float* slot = state + (size_t)seq_slots[seq] * slot_stride;
  Piece* mine = reinterpret_cast<Piece*>(e < mat ? slot + (size_t)h * mat + e : slot + (size_t)heads * mat + (size_t)h * dim + (e - mat));
  float* s_top = slot + (size_t)heads * mat + (size_t)heads * dim + (size_t)h * (tiles + 1);
  const int blocks = (len + SCAN_BLOCK - 1) / SCAN_BLOCK;
  const size_t first = (size_t)block_place(row0, seq, 0) * heads + h, width = e < mat ? mat : dim;
  float* mine_sums = (e < mat ? sums + e : norm_sums + (e - mat)) + first * width;
  const size_t stride = (size_t)heads * width;
  Piece value = fresh ? Piece(0.f) : *mine;
  float top = MODE == QIL_SCAN_MLSTM ? carried[first] : 0.f;
  const double rate = MODE == QIL_SCAN_DECAY ? (double)decay[h] : 0.0;
  const float keep_whole = MODE == QIL_SCAN_DECAY ? decay_power(rate, SCAN_BLOCK) : 0.f;   // a whole block's decay
  // eight blocks' sums are asked for before the first is taken: loads behind a store to the same array wait for nothing
  for (int c0 = 0; c0 < blocks; c0 += CARRY_AHEAD) {
    Piece add[CARRY_AHEAD];
#pragma unroll
    for (int u = 0; u < CARRY_AHEAD; ++u)
      add[u] = *reinterpret_cast<const Piece*>(mine_sums + (size_t)min(c0 + u, blocks - 1) * stride);
#pragma unroll
    for (int u = 0; u < CARRY_AHEAD; ++u) {
      const int c = c0 + u;
      if (c >= blocks) break;
      const size_t at = first + (size_t)c * heads;
      float keep, take = 1.f;
      if (MODE == QIL_SCAN_MLSTM) {
        const double local = info[at * 2], end = fmax((double)top, local);
        keep = expf((float)((double)top - end));
        take = expf((float)(local - end));
        if (e == 0) carried[at] = top;
        top = (float)(info[at * 2 + 1] + end);
      } else if (MODE == QIL_SCAN_STEP) {
        keep = expf((float)info[at * 2]);
      } else if (MODE == QIL_SCAN_CHANNEL) {
        const int last = row0 + min((c + 1) * SCAN_BLOCK, len) - 1;     // the block's last token
        keep = __builtin_amdgcn_exp2f(gsum[(size_t)last * heads * dim + (size_t)h * dim + e / vdim]);
      } else {
        const int lc = min(SCAN_BLOCK, len - c * SCAN_BLOCK);
        keep = lc == SCAN_BLOCK ? keep_whole : decay_power(rate, lc);
      }
      *reinterpret_cast<Piece*>(mine_sums + (size_t)c * stride) = value;
      value = keep * value + take * add[u];
    }
  }
  *mine = value;
  if (MODE == QIL_SCAN_MLSTM)
    for (int x = e; x < e + V && x <= tiles; ++x) s_top[x] = top;
}

// Lane t of a wave: what token t of the block weighs keys before it and the state brought in with.
template <int MODE>
__device__ __forceinline__ void outputs_weights(const float* __restrict__ gates, const float* __restrict__ gate_bias, float cap,
                                                const float* __restrict__ decay, const float* __restrict__ carried,
                                                const StepInput& steps, int h, int heads, int r0, int lc, size_t at, int lane,
                                                float* cw, float* em, float* pw, double* lead, double* tops) {
  if (MODE == QIL_SCAN_MLSTM) {
    const bool live = lane < lc;
    const GateLane g = gate_lane(gates, gate_bias, cap, r0 + (live ? lane : 0), h, heads, live, lane);
    const double brought = (double)carried[at];
    double top = g.lead;
#pragma unroll
    for (int d = 1; d < QIL_WAVE; d <<= 1) {
      const double up = __shfl_up(top, d, QIL_WAVE);
      if (lane >= d) top = fmax(top, up);
    }
    top = fmax(top, brought);
    lead[lane] = g.lead;
    tops[lane] = top;
    cw[lane] = expf((float)(brought - top));
    em[lane] = expf(-(float)(g.sum + top));
  } else if (MODE == QIL_SCAN_STEP) {
    const bool live = lane < lc;
    const StepLane g = step_lane(steps, gate_bias, decay[h], r0 + (live ? lane : 0), h, live, lane);
    tops[lane] = g.sum;
    cw[lane] = expf((float)g.sum);
    em[lane] = g.step;
  } else if (MODE != QIL_SCAN_CHANNEL) {
    pw[lane] = decay_power((double)decay[h], lane);
    if (lane == 0) pw[SCAN_BLOCK] = decay_power((double)decay[h], SCAN_BLOCK);
  }
}

// grid (blocks of the longest sequence, sequences x heads, vdim tiles)
#define OUT_SLAB 32                                               // elements of a head's dim staged at a time
#define OUT_PAD 68                                                // row of a transposed tile: 64 tokens and 4 to spread banks
template <typename T, int MODE>
__global__ void __launch_bounds__(256)
scan_outputs_kernel(const T* __restrict__ proj, int proj_row, int v_off, const float* __restrict__ qk,
                    const float* __restrict__ gates, const float* __restrict__ gate_bias, float cap,
                    const float* __restrict__ decay, const float* __restrict__ before, const float* __restrict__ norm_before,
                    const float* __restrict__ carried, const int* __restrict__ cu_seqlens, float* __restrict__ out,
                    float* __restrict__ below, int heads, int dim, int vdim, const float* __restrict__ gsum,
                    StepInput steps) {
  // first the slabs [q^T | k^T | S_in rows] (CHANNEL: and [G^T | (q 2^G)^T]), then [weighted scores^T | v]
  constexpr bool CHANNEL = MODE == QIL_SCAN_CHANNEL;
  __shared__ __align__(16) float stage[SCAN_BLOCK * OUT_PAD + SCAN_BLOCK * 64 + (CHANNEL ? 2 * OUT_SLAB * OUT_PAD : 0)];
  float* gT = stage + 2 * OUT_SLAB * OUT_PAD + OUT_SLAB * 64;
  float* eT = gT + OUT_SLAB * OUT_PAD;
  __shared__ float nin[OUT_SLAB], cw[SCAN_BLOCK], em[SCAN_BLOCK], pw[SCAN_BLOCK + 1];
  __shared__ double lead[SCAN_BLOCK], tops[SCAN_BLOCK];
  float* qT = stage;
  float* kT = stage + OUT_SLAB * OUT_PAD;
  float* sin = stage + 2 * OUT_SLAB * OUT_PAD;
  float* pT = stage;
  float* vs = stage + SCAN_BLOCK * OUT_PAD;
  const int c = blockIdx.x, seq = blockIdx.y / heads, h = blockIdx.y % heads, jt = blockIdx.z, tid = threadIdx.x;
  const int row0 = cu_seqlens[seq], len = cu_seqlens[seq + 1] - row0;
  if (c * SCAN_BLOCK >= len) return;
  const int r0 = row0 + c * SCAN_BLOCK, lc = min(SCAN_BLOCK, len - c * SCAN_BLOCK);
  const size_t at = (size_t)block_place(row0, seq, c) * heads + h;
  if (tid < QIL_WAVE)
    outputs_weights<MODE>(gates, gate_bias, cap, decay, carried, steps, h, heads, r0, lc, at, tid, cw, em, pw, lead, tops);
  const int ti = tid / 16, tj = tid % 16;
  const size_t hd = (size_t)heads * dim;
  const int group = MODE == QIL_SCAN_STEP ? h / (heads / steps.groups) : h;
  const float* s_in = before + at * dim * vdim;
  float p[4][4] = {}, o[4][4] = {}, nq[4] = {};
  for (int i0 = 0; i0 < dim; i0 += OUT_SLAB) {
    __syncthreads();
    for (int idx = tid; idx < SCAN_BLOCK * OUT_SLAB; idx += 256) {
      const int t = idx / OUT_SLAB, x = idx % OUT_SLAB, i = i0 + x;
      const bool ok = t < lc && i < dim;
      if (MODE == QIL_SCAN_STEP) {
        const T* row = proj + (size_t)(r0 + (ok ? t : 0)) * proj_row + group * dim + (ok ? i : 0);
        qT[x * OUT_PAD + t] = ok ? ld(row + steps.q_off) : 0.f;
        kT[x * OUT_PAD + t] = ok ? ld(row + steps.k_off) : 0.f;
        continue;
      }
      const float* src = qk + (size_t)(r0 + (ok ? t : 0)) * 2 * hd + (size_t)h * dim + (ok ? i : 0);
      qT[x * OUT_PAD + t] = ok ? src[0] : 0.f;
      kT[x * OUT_PAD + t] = ok ? src[hd] : 0.f;
      if (CHANNEL) {
        const float g = ok ? gsum[(size_t)(r0 + t) * hd + (size_t)h * dim + i] : 0.f;
        gT[x * OUT_PAD + t] = g;
        eT[x * OUT_PAD + t] = ok ? src[0] * __builtin_amdgcn_exp2f(g) : 0.f;
      }
    }
    for (int idx = tid; idx < OUT_SLAB * 64; idx += 256) {
      const int x = idx / 64, y = idx % 64, i = i0 + x, j = jt * 64 + y;
      sin[x * 64 + y] = (i < dim && j < vdim) ? s_in[(size_t)i * vdim + j] : 0.f;
    }
    if (MODE == QIL_SCAN_MLSTM && tid < OUT_SLAB) nin[tid] = i0 + tid < dim ? norm_before[at * dim + i0 + tid] : 0.f;
    __syncthreads();
#pragma unroll 4
    for (int x = 0; x < OUT_SLAB; ++x) {
      const float4 q4 = *reinterpret_cast<const float4*>(&qT[x * OUT_PAD + ti * 4]);
      const float4 k4 = *reinterpret_cast<const float4*>(&kT[x * OUT_PAD + tj * 4]);
      const float4 s4 = *reinterpret_cast<const float4*>(&sin[x * 64 + tj * 4]);
      const float q[4] = {q4.x, q4.y, q4.z, q4.w}, k[4] = {k4.x, k4.y, k4.z, k4.w}, s[4] = {s4.x, s4.y, s4.z, s4.w};
      const float nx = MODE == QIL_SCAN_MLSTM ? nin[x] : 0.f;
      if (CHANNEL) {
        // the weight 2^(G_t - G_s) of every (query, key, row of S) inside the sum; what came in is taken by q 2^G_t
        const float4 e4 = *reinterpret_cast<const float4*>(&eT[x * OUT_PAD + ti * 4]);
        const float qe[4] = {e4.x, e4.y, e4.z, e4.w};
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int u = 0; u < 4; ++u) o[r][u] += qe[r] * s[u];
        if (tj <= ti) {                                          // (tiles above the diagonal hold no visible key)
          const float4 a4 = *reinterpret_cast<const float4*>(&gT[x * OUT_PAD + ti * 4]);
          const float4 b4 = *reinterpret_cast<const float4*>(&gT[x * OUT_PAD + tj * 4]);
          const float gt[4] = {a4.x, a4.y, a4.z, a4.w}, gs[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
          for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int u = 0; u < 4; ++u) p[r][u] += q[r] * k[u] * __builtin_amdgcn_exp2f(fminf(gt[r] - gs[u], 0.f));
        }
        continue;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          p[r][u] += q[r] * k[u];
          o[r][u] += q[r] * s[u];
        }
        if (MODE == QIL_SCAN_MLSTM) nq[r] += q[r] * nx;
      }
    }
  }
  // the weights: scores of keys at or before the token by exp(e_s - M_t), what came in by exp(m_in - M_t)
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int t = ti * 4 + r;
    const float brought = (MODE == QIL_SCAN_MLSTM || MODE == QIL_SCAN_STEP) ? cw[t] : CHANNEL ? 1.f : pw[t + 1];
    float row_sum = 0.f;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int s = tj * 4 + u;
      float weight = 0.f;
      if (s <= t && t < lc)
        weight = MODE == QIL_SCAN_MLSTM ? expf((float)(lead[s] - tops[t]))
                 : MODE == QIL_SCAN_STEP ? expf((float)(tops[t] - tops[s])) * em[s]
                 : CHANNEL ? 1.f : pw[t - s];
      p[r][u] *= weight;
      row_sum += p[r][u];
      o[r][u] *= brought;
    }
    if (MODE == QIL_SCAN_MLSTM) {
      row_sum += __shfl_xor(row_sum, 1, QIL_WAVE);
      row_sum += __shfl_xor(row_sum, 2, QIL_WAVE);
      row_sum += __shfl_xor(row_sum, 4, QIL_WAVE);
      row_sum += __shfl_xor(row_sum, 8, QIL_WAVE);
      nq[r] = nq[r] * brought + row_sum;
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < 4; ++u)
    *reinterpret_cast<float4*>(&pT[(tj * 4 + u) * OUT_PAD + ti * 4]) = make_float4(p[0][u], p[1][u], p[2][u], p[3][u]);
  for (int idx = tid; idx < SCAN_BLOCK * 64; idx += 256) {
    const int s = idx / 64, y = idx % 64, j = jt * 64 + y;
    vs[s * 64 + y] = (s < lc && j < vdim) ? ld(proj + (size_t)(r0 + s) * proj_row + v_off + h * vdim + j) : 0.f;
  }
  __syncthreads();
  for (int s = 0; s < lc; ++s) {
    const float4 p4 = *reinterpret_cast<const float4*>(&pT[s * OUT_PAD + ti * 4]);
    const float4 v4 = *reinterpret_cast<const float4*>(&vs[s * 64 + tj * 4]);
    const float a[4] = {p4.x, p4.y, p4.z, p4.w}, b[4] = {v4.x, v4.y, v4.z, v4.w};
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int u = 0; u < 4; ++u) o[r][u] += a[r] * b[u];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int t = ti * 4 + r;
    if (t >= lc) continue;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = jt * 64 + tj * 4 + u;
      if (j < vdim) out[(size_t)(r0 + t) * heads * vdim + (size_t)h * vdim + j] = o[r][u];
    }
    if (MODE == QIL_SCAN_MLSTM && jt == 0 && tj == 0) below[(size_t)(r0 + t) * heads + h] = fmaxf(fabsf(nq[r]), em[t]) + 1e-6f;
  }
}

// ---- DECAY and MLSTM on the matrix cores: dim 64, 128 or 256, vdim a multiple of 64, values in aligned pairs.
// v_mfma_f32_32x32x2_f32 takes float32 inputs and adds float32 products into float32 sums, as the vector units do, at twice
// their rate; what bounds the kernels above is their LDS reads (three 16-byte reads for 16 or 32 multiplications).  The index
// that a product sums over may be numbered as one likes: step u of group g takes tokens (or state rows) 8 g + u and
// 8 g + 4 + u, so that a lane's four steps are four neighbours in memory.  Columns are paired the same way (tile j takes
// the columns 2 lane + j), so that state, values and results move as 8-byte pieces in whole lines, straight between
// memory and registers.
typedef float scan_x16 __attribute__((ext_vector_type(16)));
__device__ __forceinline__ scan_x16 scan_mfma(float a, float b, scan_x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
// row of result register r (of 16) in a 32 x 32 tile, lane half `up`
__device__ __forceinline__ int scan_tile_row(int r, int up) { return 8 * (r / 4) + 4 * up + r % 4; }

// Two neighbouring values as they lie in memory, and as floats.
template <typename T> struct ValuePair;
template <> struct ValuePair<float> {
  float2 raw;
  __device__ __forceinline__ void load(const float* p) { raw = *reinterpret_cast<const float2*>(p); }
  __device__ __forceinline__ float at(int i, bool live) const { return live ? (i ? raw.y : raw.x) : 0.f; }
};
template <> struct ValuePair<bf16_t> {
  uint32_t raw;
  __device__ __forceinline__ void load(const bf16_t* p) { raw = *reinterpret_cast<const uint32_t*>(p); }
  __device__ __forceinline__ float at(int i, bool live) const {
    return live ? __uint_as_float(i ? raw & 0xffff0000u : raw << 16) : 0.f;
  }
};

// As scan_sums_kernel.  A wave makes 64 rows by 64 columns of a block's sum over its 64 tokens, 128 products; keys and values
// come straight from memory (a block's waves share the keys).  grid (blocks of the longest sequence, sequences x heads, dim
// tiles x groups of column tiles); blockDim.x / 64 column tiles a group.
template <typename T, int MODE>
__global__ void __launch_bounds__(256)
scan_sums_mfma_kernel(const T* __restrict__ proj, int proj_row, int v_off, const float* __restrict__ qk,
                      const float* __restrict__ gates, const float* __restrict__ gate_bias, float cap,
                      const float* __restrict__ decay, const float* __restrict__ state, size_t slot_stride,
                      const int* __restrict__ cu_seqlens, const int* __restrict__ seq_starts, const int* __restrict__ seq_slots,
                      float* __restrict__ sums, float* __restrict__ norm_sums, double* __restrict__ info,
                      float* __restrict__ carried, int heads, int dim, int vdim, int dim_tiles) {
  __shared__ __align__(16) float w[SCAN_BLOCK];
  const int c = blockIdx.x, seq = blockIdx.y / heads, h = blockIdx.y % heads, tid = threadIdx.x;
  const int it = blockIdx.z % dim_tiles, jt = blockIdx.z / dim_tiles * (blockDim.x / QIL_WAVE) + tid / QIL_WAVE;
  const int lane = tid % QIL_WAVE, up = lane / 32, col = lane % 32;
  const int row0 = cu_seqlens[seq], len = cu_seqlens[seq + 1] - row0;
  if (c * SCAN_BLOCK >= len) return;
  const int r0 = row0 + c * SCAN_BLOCK, lc = min(SCAN_BLOCK, len - c * SCAN_BLOCK);
  const size_t at = (size_t)block_place(row0, seq, c) * heads + h, hd = (size_t)heads * dim;
  const float* keys = qk + hd + (size_t)h * dim + it * 64 + 2 * col;
  const T* values = proj + v_off + h * vdim + jt * 64 + 2 * col;
  constexpr int AHEAD = 2;
  float2 k[AHEAD][4];
  ValuePair<T> v[AHEAD][4];
  auto ask = [&](int g, int slot) {                              // tokens past the block's end read its last one
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const size_t row = r0 + min(8 * g + 4 * up + u, lc - 1);
      k[slot][u] = *reinterpret_cast<const float2*>(keys + row * 2 * hd);
      v[slot][u].load(values + row * proj_row);
    }
  };
#pragma unroll
  for (int g = 0; g < AHEAD; ++g) ask(g, g);
  StepInput none{};
  if (tid < QIL_WAVE)
    w[tid] = sums_weight<MODE>(gates, gate_bias, cap, decay, state, slot_stride, seq_starts, seq_slots, info, carried, heads,
                               dim, vdim, none, seq, h, c, r0, lc, at, blockIdx.z == 0, tid);
  __syncthreads();
  scan_x16 acc[2][2] = {};
  float norm[2] = {};
#pragma unroll
  for (int g = 0; g < SCAN_BLOCK / 8; ++g) {
    const float4 w4 = *reinterpret_cast<const float4*>(&w[8 * g + 4 * up]);
    const float weight[4] = {w4.x, w4.y, w4.z, w4.w};
    float a[2][4], b[2][4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool live = 8 * g + 4 * up + u < lc;
      a[0][u] = live ? weight[u] * k[g % AHEAD][u].x : 0.f;
      a[1][u] = live ? weight[u] * k[g % AHEAD][u].y : 0.f;
      b[0][u] = v[g % AHEAD][u].at(0, live);
      b[1][u] = v[g % AHEAD][u].at(1, live);
    }
    if (g + AHEAD < SCAN_BLOCK / 8) ask(g + AHEAD, g % AHEAD);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (MODE == QIL_SCAN_MLSTM) norm[i] += a[i][u];
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = scan_mfma(a[i][u], b[j][u], acc[i][j]);
      }
    }
  }
  float* to = sums + at * dim * vdim + (size_t)it * 64 * vdim + jt * 64 + 2 * col;
#pragma unroll
  for (int r = 0; r < 16; ++r)
#pragma unroll
    for (int i = 0; i < 2; ++i)
      *reinterpret_cast<float2*>(to + (size_t)(2 * scan_tile_row(r, up) + i) * vdim) = make_float2(acc[i][0][r], acc[i][1][r]);
  if (MODE == QIL_SCAN_MLSTM && jt == 0) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const float total = norm[i] + __shfl_xor(norm[i], 32, QIL_WAVE);
      if (up == 0) norm_sums[at * dim + it * 64 + 2 * col + i] = total;
    }
  }
}

// As scan_outputs_kernel: a block makes 64 tokens by 64 columns a wave.  Queries and keys pass through LDS (rows of DIM + 4
// floats: 16 lanes' 16-byte reads fall on all 64 banks), the state brought in and the values come straight from memory.  The
// scores are made once a block (the kernel above makes them for every 64 columns again), the quadrant of keys behind the
// tokens not at all; the weighted scores take the keys' place in LDS.  grid (blocks of the longest sequence, sequences x
// heads, groups of column tiles).
template <typename T, int MODE, int DIM>
__global__ void __launch_bounds__(256, DIM <= 128 ? 2 : 1)
scan_outputs_mfma_kernel(const T* __restrict__ proj, int proj_row, int v_off, const float* __restrict__ qk,
                         const float* __restrict__ gates, const float* __restrict__ gate_bias, float cap,
                         const float* __restrict__ decay, const float* __restrict__ before,
                         const float* __restrict__ norm_before, const float* __restrict__ carried,
                         const int* __restrict__ cu_seqlens, float* __restrict__ out, float* __restrict__ below, int heads,
                         int vdim) {
  constexpr int ROW = DIM + 4, PROW = SCAN_BLOCK + 4, GROUPS = DIM / 8, AHEAD = MODE == QIL_SCAN_MLSTM ? 2 : 3, VALUES = 2;
  extern __shared__ __align__(16) float scan_lds[];
  float* qs = scan_lds;                                          // [64][ROW]
  float* ks = scan_lds + SCAN_BLOCK * ROW;                       // [64][ROW], later the weighted scores [64][PROW]
  float* ps = ks;
  __shared__ __align__(16) float cw[SCAN_BLOCK], em[SCAN_BLOCK], pw[SCAN_BLOCK + 1];
  __shared__ double lead[SCAN_BLOCK], tops[SCAN_BLOCK];
  const int c = blockIdx.x, seq = blockIdx.y / heads, h = blockIdx.y % heads, tid = threadIdx.x;
  const int waves = blockDim.x / QIL_WAVE, wave = tid / QIL_WAVE, lane = tid % QIL_WAVE, up = lane / 32, col = lane % 32;
  const int row0 = cu_seqlens[seq], len = cu_seqlens[seq + 1] - row0;
  if (c * SCAN_BLOCK >= len) return;
  const int r0 = row0 + c * SCAN_BLOCK, lc = min(SCAN_BLOCK, len - c * SCAN_BLOCK);
  const size_t at = (size_t)block_place(row0, seq, c) * heads + h, hd = (size_t)heads * DIM;
  const int j0 = (blockIdx.z * waves + wave) * 64 + 2 * col;
  const float* s_in = before + at * DIM * vdim + (size_t)4 * up * vdim + j0;
  float2 s[AHEAD][4];
  auto ask_state = [&](int g, int slot) {
#pragma unroll
    for (int u = 0; u < 4; ++u) s[slot][u] = *reinterpret_cast<const float2*>(s_in + (size_t)(8 * g + u) * vdim);
  };
  {                                                              // queries and keys into LDS, rows past the end as zeros
    const float* src = qk + (size_t)r0 * 2 * hd + (size_t)h * DIM;
#pragma unroll 8
    for (int idx = tid; idx < 2 * SCAN_BLOCK * (DIM / 4); idx += blockDim.x) {
      const int x = idx % (DIM / 4), t = idx / (DIM / 4) % SCAN_BLOCK, key = idx / (DIM / 4) / SCAN_BLOCK;
      float4 q = *reinterpret_cast<const float4*>(src + (size_t)min(t, lc - 1) * 2 * hd + key * hd + 4 * x);
      if (t >= lc) q = make_float4(0.f, 0.f, 0.f, 0.f);
      *reinterpret_cast<float4*>(&qs[(key * SCAN_BLOCK + t) * ROW + 4 * x]) = q;
    }
  }
#pragma unroll
  for (int g = 0; g < AHEAD; ++g) ask_state(g, g);
  StepInput none{};
  if (tid < QIL_WAVE)
    outputs_weights<MODE>(gates, gate_bias, cap, decay, carried, none, h, heads, r0, lc, at, tid, cw, em, pw, lead, tops);
  __syncthreads();
  scan_x16 o[2][2] = {};
#pragma unroll
  for (int g = 0; g < GROUPS; ++g) {
    float a[2][4], b[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const float4 q = *reinterpret_cast<const float4*>(&qs[(32 * t + col) * ROW + 8 * g + 4 * up]);
      a[t][0] = q.x; a[t][1] = q.y; a[t][2] = q.z; a[t][3] = q.w;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) { b[0][u] = s[g % AHEAD][u].x; b[1][u] = s[g % AHEAD][u].y; }
    if (g + AHEAD < GROUPS) ask_state(g + AHEAD, g % AHEAD);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < 2; ++j) o[t][j] = scan_mfma(a[t][u], b[j][u], o[t][j]);
  }
  const T* values = proj + v_off + h * vdim + j0;
  ValuePair<T> v[VALUES][4];
  auto ask_values = [&](int g, int slot) {
#pragma unroll
    for (int u = 0; u < 4; ++u)
      v[slot][u].load(values + (size_t)(r0 + min(8 * g + 4 * up + u, lc - 1)) * proj_row);
  };
#pragma unroll
  for (int g = 0; g < VALUES; ++g) ask_values(g, g);
  // the state's part by what a token weighs it with
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int token = 32 * t + scan_tile_row(r, up);
      const float brought = MODE == QIL_SCAN_MLSTM ? cw[token] : pw[token + 1];
      o[t][0][r] *= brought;
      o[t][1][r] *= brought;
    }
  // the scores' three quadrants, one a wave where there are four waves: tokens from 32 (n > 0), keys from 32 (n > 1)
  scan_x16 p[3];
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const int n = wave + m * waves;
    if (n >= 3) continue;
    p[m] = scan_x16{};
    const float* a_row = &qs[((n > 0 ? 32 : 0) + col) * ROW + 4 * up];
    const float* b_row = &ks[((n > 1 ? 32 : 0) + col) * ROW + 4 * up];
#pragma unroll 8
    for (int g = 0; g < GROUPS; ++g) {
      const float4 a = *reinterpret_cast<const float4*>(a_row + 8 * g), b = *reinterpret_cast<const float4*>(b_row + 8 * g);
      p[m] = scan_mfma(a.x, b.x, p[m]);
      p[m] = scan_mfma(a.y, b.y, p[m]);
      p[m] = scan_mfma(a.z, b.z, p[m]);
      p[m] = scan_mfma(a.w, b.w, p[m]);
    }
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    const int n = wave + m * waves, key = (n > 1 ? 32 : 0) + col;
    if (n >= 3) continue;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int token = (n > 0 ? 32 : 0) + scan_tile_row(r, up);
      float value = 0.f;
      if (key <= token && token < lc)
        value = p[m][r] * (MODE == QIL_SCAN_MLSTM ? expf((float)(lead[key] - tops[token])) : pw[max(token - key, 0)]);
      ps[token * PROW + key] = value;
    }
  }
  __syncthreads();
  if (MODE == QIL_SCAN_MLSTM && blockIdx.z == 0 && wave == waves - 1 && lane < lc) {
    const float* n_in = norm_before + at * DIM;
    float dot = 0.f, row_sum = 0.f;
#pragma unroll 2
    for (int x = 0; x < DIM; x += 4) {
      const float4 q = *reinterpret_cast<const float4*>(&qs[lane * ROW + x]);
      dot += q.x * n_in[x];
      dot += q.y * n_in[x + 1];
      dot += q.z * n_in[x + 2];
      dot += q.w * n_in[x + 3];
    }
    for (int x = 0; x <= lane; ++x) row_sum += ps[lane * PROW + x];
    below[(size_t)(r0 + lane) * heads + h] = fmaxf(fabsf(dot * cw[lane] + row_sum), em[lane]) + 1e-6f;
  }
#pragma unroll
  for (int g = 0; g < SCAN_BLOCK / 8; ++g) {
    float a[2][4], b[2][4];
#pragma unroll
    for (int t = g < 4 ? 0 : 1; t < 2; ++t) {                    // the first 32 tokens see none of the last 32 keys
      const float4 q = *reinterpret_cast<const float4*>(&ps[(32 * t + col) * PROW + 8 * g + 4 * up]);
      a[t][0] = q.x; a[t][1] = q.y; a[t][2] = q.z; a[t][3] = q.w;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const bool live = 8 * g + 4 * up + u < lc;
      b[0][u] = v[g % VALUES][u].at(0, live);
      b[1][u] = v[g % VALUES][u].at(1, live);
    }
    if (g + VALUES < SCAN_BLOCK / 8) ask_values(g + VALUES, g % VALUES);
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int t = g < 4 ? 0 : 1; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < 2; ++j) o[t][j] = scan_mfma(a[t][u], b[j][u], o[t][j]);
  }
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int token = 32 * t + scan_tile_row(r, up);
      if (token < lc)
        *reinterpret_cast<float2*>(out + (size_t)(r0 + token) * heads * vdim + (size_t)h * vdim + j0) =
            make_float2(o[t][0][r], o[t][1][r]);
    }
}

// What the two kernels above take: whole tiles, and rows whose pairs of values are aligned.
static bool scan_mfma_takes(const void* proj, int dtype, int proj_row, int v_off, const float* workspace, const float* out,
                            int dim, int vdim) {
  return (dim == 64 || dim == 128 || dim == 256) && vdim % 64 == 0 && proj_row % 2 == 0 && v_off % 2 == 0 &&
         (uintptr_t)proj % (dtype == QIL_F32 ? 8 : 4) == 0 && (uintptr_t)workspace % 16 == 0 && (uintptr_t)out % 8 == 0;
}

template <typename T, int MODE, int DIM>
static int scan_outputs_mfma(dim3 grid, int threads, const T* proj, int proj_row, int v_off, const float* qk,
                             const float* gates, const float* gate_bias, float cap, const float* decay, const float* before,
                             const float* norm_before, const float* carried, const int* cu_seqlens, float* out, float* below,
                             int heads, int vdim, hipStream_t s) {
  constexpr size_t lds = 2 * SCAN_BLOCK * (DIM + 4) * sizeof(float);
  if (lds > 64 * 1024) {
    static bool granted = false;
    if (!granted) {
      hipError_t e = hipFuncSetAttribute((const void*)scan_outputs_mfma_kernel<T, MODE, DIM>,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
      if (e != hipSuccess) return (int)e;
      granted = true;
    }
  }
  hipLaunchKernelGGL((scan_outputs_mfma_kernel<T, MODE, DIM>), grid, dim3(threads), lds, s, proj, proj_row, v_off, qk, gates,
                     gate_bias, cap, decay, before, norm_before, carried, cu_seqlens, out, below, heads, vdim);
  return 0;
}

static size_t chunked_places(int n, int n_seqs) { return (size_t)n / SCAN_BLOCK + n_seqs; }

extern "C" {

// Floats of the scratch memory of a step of n rows in n_seqs sequences.
size_t qil_state_scan_chunked_workspace(int n, int n_seqs, int heads, int dim, int vdim, int mode) {
  const size_t places = chunked_places(n, n_seqs);
  size_t floats = places * heads * 4 + (places * heads + 3) / 4 * 4 + places * heads * dim * vdim;
  if (mode != QIL_SCAN_STEP) floats += (size_t)n * 2 * heads * dim;
  if (mode == QIL_SCAN_MLSTM) floats += places * heads * dim;
  if (mode == QIL_SCAN_CHANNEL) floats += (size_t)n * heads * dim;
  return floats;
}

// As qil_state_scan, for steps in which a sequence has many rows (max_query: the most rows of one sequence).
int qil_state_scan_chunked(const void* proj, int dtype, int proj_row, int q_off, int k_off, int v_off, const float* gates,
                           const float* gate_bias, float cap, const float* decay, const float* freq, int rot, float q_scale,
                           float k_scale, float* state, size_t slot_stride, const int* cu_seqlens, const int* seq_starts,
                           const int* seq_slots, float* out, float* below, float* workspace, int n, int n_seqs,
                           int max_query, int heads, int dim, int vdim, int mode, const void* raw, int raw_code,
                           int raw_splits, int raw_row, int groups, hipStream_t s) {
  if (n_seqs == 0 || n == 0) return 0;
  if (dim < 1 || vdim < 1 || rot < 0 || rot % 2 || rot > dim || max_query < 1 ||
      mode < QIL_SCAN_DECAY || mode > QIL_SCAN_STEP || !workspace || (size_t)n_seqs * heads > 65535)
    return -1;
  if ((mode == QIL_SCAN_MLSTM && (!gates || !gate_bias || !below)) || (mode == QIL_SCAN_DECAY && !decay) ||
      (mode == QIL_SCAN_CHANNEL && (!gates || !(cap > 0.f) || n_seqs > 65535)) || (rot && !freq)) return -1;
  if (mode == QIL_SCAN_STEP && (!raw || !gate_bias || !decay || groups < 1 || heads % groups || rot || raw_splits < 1 ||
                                (raw_code == QIL_BF16 && raw_splits != 1) || raw_row < heads)) return -1;
  const StepInput steps{{raw, raw_code, raw_splits, (size_t)n * raw_row}, raw_row, q_off, k_off, groups};
  const size_t places = chunked_places(n, n_seqs);
  double* info = reinterpret_cast<double*>(workspace);
  float* carried = workspace + places * heads * 4;
  float* qk = carried + (places * heads + 3) / 4 * 4;
  float* sums = qk + (mode == QIL_SCAN_STEP ? 0 : (size_t)n * 2 * heads * dim);
  float* norm_sums = sums + places * heads * dim * vdim;
  float* gsum = norm_sums;                                       // CHANNEL has no normaliser: its place holds the decays' sums
  const int blocks = (max_query + SCAN_BLOCK - 1) / SCAN_BLOCK;
  const int dim_tiles = (dim + 63) / 64, v_tiles = (vdim + 63) / 64;
  const int per_head = dim * vdim + (mode == QIL_SCAN_MLSTM ? dim : 0);
  const bool quads = dim % 4 == 0 && vdim % 4 == 0 && slot_stride % 4 == 0 &&
                     ((uintptr_t)state | (uintptr_t)workspace) % 16 == 0;
  const bool matrix_cores = scan_mfma_takes(proj, dtype, proj_row, v_off, workspace, out, dim, vdim);
  const dim3 g_sums(blocks, n_seqs * heads, dim_tiles * v_tiles);
  const dim3 g_out(blocks, n_seqs * heads, v_tiles);
  const int units = dim - rot / 2;                               // pairs and single elements of a head that rotate works on
#define QIL_CARRY(MODE)                                                                                               \
  if (quads)                                                                                                          \
    hipLaunchKernelGGL((scan_carry_kernel<MODE, 4>), dim3(n_seqs, heads, (per_head / 4 + 255) / 256), dim3(256), 0, s,  \
                       sums, norm_sums, info, carried, decay, state, slot_stride, cu_seqlens, seq_starts, seq_slots,   \
                       heads, dim, vdim, gsum);                                                                       \
  else                                                                                                                \
    hipLaunchKernelGGL((scan_carry_kernel<MODE, 1>), dim3(n_seqs, heads, (per_head + 255) / 256), dim3(256), 0, s,     \
                       sums, norm_sums, info, carried, decay, state, slot_stride, cu_seqlens, seq_starts, seq_slots,   \
                       heads, dim, vdim, gsum)
#define QIL_CHUNKED(T, MODE)                                                                                          \
  do {                                                                                                                \
    if (MODE == QIL_SCAN_CHANNEL)                                                                                     \
      hipLaunchKernelGGL(scan_decays_kernel, dim3(blocks, n_seqs, (heads * dim + 255) / 256), dim3(256), 0, s, gates,  \
                         cap, cu_seqlens, gsum, heads * dim);                                                          \
    if (MODE != QIL_SCAN_STEP)                                                                                        \
      hipLaunchKernelGGL(scan_rotate_kernel<T>, dim3(n), dim3(256 / units * units), 0, s, (const T*)proj, proj_row,    \
                         q_off, k_off, freq, rot, q_scale, k_scale, cu_seqlens, seq_starts, n_seqs, qk, heads, dim);   \
    if constexpr (MODE == QIL_SCAN_DECAY || MODE == QIL_SCAN_MLSTM)                                                   \
      if (matrix_cores) {                                                                                             \
        const int waves = v_tiles % 4 == 0 ? 4 : v_tiles % 2 == 0 ? 2 : 1;                                            \
        hipLaunchKernelGGL((scan_sums_mfma_kernel<T, MODE>), dim3(blocks, n_seqs * heads, dim_tiles * v_tiles / waves), \
                           dim3(waves * QIL_WAVE), 0, s, (const T*)proj, proj_row, v_off, qk, gates, gate_bias, cap,   \
                           decay, state, slot_stride, cu_seqlens, seq_starts, seq_slots, sums, norm_sums, info, carried, \
                           heads, dim, vdim, dim_tiles);                                                              \
        QIL_CARRY(MODE);                                                                                              \
        const auto outputs = dim == 64    ? scan_outputs_mfma<T, MODE, 64>                                            \
                             : dim == 128 ? scan_outputs_mfma<T, MODE, 128>                                           \
                                          : scan_outputs_mfma<T, MODE, 256>;                                          \
        const int status = outputs(dim3(blocks, n_seqs * heads, v_tiles / waves), waves * QIL_WAVE, (const T*)proj,    \
                                   proj_row, v_off, qk, gates, gate_bias, cap, decay, sums, norm_sums, carried,        \
                                   cu_seqlens, out, below, heads, vdim, s);                                           \
        if (status) return status;                                                                                    \
        break;                                                                                                        \
      }                                                                                                               \
    hipLaunchKernelGGL((scan_sums_kernel<T, MODE>), g_sums, dim3(256), 0, s, (const T*)proj, proj_row, v_off, qk,      \
                       gates, gate_bias, cap, decay, state, slot_stride, cu_seqlens, seq_starts, seq_slots, sums,      \
                       norm_sums, info, carried, heads, dim, vdim, dim_tiles, gsum, steps);                            \
    QIL_CARRY(MODE);                                                                                                  \
    hipLaunchKernelGGL((scan_outputs_kernel<T, MODE>), g_out, dim3(256), 0, s, (const T*)proj, proj_row, v_off, qk,    \
                       gates, gate_bias, cap, decay, sums, norm_sums, carried, cu_seqlens, out, below, heads, dim,     \
                       vdim, gsum, steps);                                                                             \
  } while (0)
  if (dtype == QIL_F32) {
    if (mode == QIL_SCAN_MLSTM) QIL_CHUNKED(float, QIL_SCAN_MLSTM);
    else if (mode == QIL_SCAN_CHANNEL) QIL_CHUNKED(float, QIL_SCAN_CHANNEL);
    else if (mode == QIL_SCAN_STEP) QIL_CHUNKED(float, QIL_SCAN_STEP);
    else QIL_CHUNKED(float, QIL_SCAN_DECAY);
  } else {
    if (mode == QIL_SCAN_MLSTM) QIL_CHUNKED(bf16_t, QIL_SCAN_MLSTM);
    else if (mode == QIL_SCAN_CHANNEL) QIL_CHUNKED(bf16_t, QIL_SCAN_CHANNEL);
    else if (mode == QIL_SCAN_STEP) QIL_CHUNKED(bf16_t, QIL_SCAN_STEP);
    else QIL_CHUNKED(bf16_t, QIL_SCAN_DECAY);
  }
#undef QIL_CHUNKED
#undef QIL_CARRY
  QIL_RETURN_LAUNCH_STATUS();
}

}  // extern "C"
