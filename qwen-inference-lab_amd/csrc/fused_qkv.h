// What a decode attention kernel needs to make its queries, the new key and the new value itself (attention_decode.hip,
// attention_decode_f32.hip).
#pragma once

// FUSED: the queries do not come from memory but from the partial sums of the q/k/v product, with the
// head norm and the rotation made here (the arithmetic of qk_rope.hip, shared through qk_math.h); and the
// wave that meets the row's own position makes the new key and value the same way, writes them into the
// pages and uses them from its registers.  One kernel less per layer in a decode step.
struct FusedQKV {
  const float* qkv;                                        // [splits][rows][(heads + 2 kv_heads) d] partial sums
  size_t split_stride;
  int splits;
  const float* q_weight;                                   // null: no head norm
  const float* k_weight;
  float eps;
  const float* cos_table;                                  // null: no rotation
  const float* sin_table;                                  // null with a cos_table: that holds rot / 2 frequencies
  int rot;
  int rotate_first;                                        // the rotation comes before the head norm
  int writes;                                              // 0: the cache belongs to another layer, which wrote it
  int row_elems;                                           // elements of a row of qkv (more than q, k and v where another
                                                           // branch's columns follow; q alone for a reader without k and v)
  int v_head;                                              // the head-sized piece of a row at which the values begin
                                                           // (heads + kv_heads; heads: the values are the keys before norm
                                                           // and rotation)
  const float* bias;                                       // null, or the projection's bias by column, added to the sums
  float temp_coef;                                         // temp_every > 0: the query at position p is multiplied by
  int temp_every;                                          // 1 + temp_coef * ln(floor((p + 1) / temp_every) + 1) last
};

// Reads the fields at a kernel's start, all with one wait: where each is read at its use, a wave waits for a dozen of them in
// turn before its first load of data.
__device__ __forceinline__ void ask_fields(const FusedQKV& f) {
  asm volatile("" ::"s"(f.qkv), "s"(f.split_stride), "s"(f.splits), "s"(f.q_weight), "s"(f.k_weight), "s"(f.eps), "s"(f.cos_table),
               "s"(f.sin_table), "s"(f.rot), "s"(f.rotate_first), "s"(f.writes), "s"(f.row_elems), "s"(f.v_head), "s"(f.bias),
               "s"(f.temp_coef), "s"(f.temp_every));
}
