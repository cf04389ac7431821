// How many queries a tile of each attention kernel's work list holds: the one place where these
// sizes are written.  The kernels include it; who makes the lists asks eng_attn_tile_sizes().
#pragma once

// The optional terms of a score and of the output that the attention kernels' `_terms` entry
// points take (a null pointer or 0 where a term is absent).  A score is made in this order:
//   s = (q . k) * scale            (head_scale[h] instead of scale where given)
//   s = softcap * tanh(s / softcap)                       (softcap > 0)
//   s -= slopes[h] * (query position - key position)
//   s += dist_bias[h * n_dist + min(distance, n_dist - 1)]      (a table of float, a row a head)
// keep_first: with a window, the first so many keys stay visible.  gate (rows of stride ldg, the
// queries' element type): the output is multiplied by its sigmoid.  sinks [n_heads]: the softmax's
// denominator holds exp(sinks[h]) too, a number beside the scores that brings no value.  head_gate
// (float rows of stride ldhg, a column a head): head h's output is multiplied by the sigmoid of its
// column.
struct AttnTerms {
  const float* head_scale;
  const float* slopes;
  const void* gate;
  int ldg, keep_first;
  float softcap;
  const float* dist_bias;
  int n_dist;
  const float* sinks;
  const float* head_gate;
  int ldhg;
};

#ifdef __HIPCC__
// From l = the sum of exp(score - m) over the keys to the whole denominator (m the largest score).
template <typename Args>
__device__ __forceinline__ float with_sink(const Args& p, int h, float m, float l) {
  return p.sinks ? l + expf(p.sinks[h] - m) : l;
}
template <typename Args>
__device__ __forceinline__ float head_gate_of(const Args& p, int row, int h) {
  return p.head_gate ? 1.0f / (1.0f + expf(-p.head_gate[(size_t)row * p.ldhg + h])) : 1.0f;
}
#endif

#define ATTN_TILE_QUERIES 16           // attn_tile (attention.hip): queries a block
#define ATTN_PREFILL_TILE_QUERIES 128  // attn_prefill (attention_prefill.hip): queries a block

// How the decode kernel (attention_decode.hip) is launched for n_rows single rows of n_heads
// heads whose longest walk is `keys` keys (a window's and its kept first keys' at most): in how
// many parts a row's keys go at most, and the waves a block.
// Eight waves a block; four where the rows' blocks alone are more than the CUs (64 rows of 25 heads
// at contexts of 300 to 1,001: 49.2 us, 49.7 with eight, 53.5 with two; 24 rows 20.4 and 22.6), or the keys no
// more than four waves' tiles; sixteen where blocks that have a CU each may walk 2,048 keys or more (8 rows at
// 4,000 to 8,001: 57.1 us, 59.3 with eight).  A recorded step is planned for its class's longest, and a row of fewer
// than ATTN_DECODE_WIDE_ROW_FROM keys lets its block's second eight waves end (8 rows of 25 heads of 64 at 60 to 500
// keys: 9.1 us with sixteen, 8.4 with eight; 500 to 900 12.0 and 11.4; 900 to 1,300 15.1 and 14.6, of 6 rows 13.9 and
// 14.2; 1,300 to 1,900 of 6 rows 17.4 and 18.2).  Splits only where a wave would walk 64 keys or more, as many as
// leave it 32, and no more than give every block a compute unit at once (one row at 700 keys: 8.1 us in two, 8.7
// whole; at 6,000: 13.4 in eight).
#define ATTN_DECODE_ROW_WAVES 8
#define ATTN_DECODE_WIDE_ROW_FROM 1024
#define ATTN_DECODE_TILE_KEYS 16
#define ATTN_DECODE_SPLIT_KEYS_A_WAVE 64
#define ATTN_DECODE_KEYS_A_PART 32
static inline void attn_decode_row_work(int n_compute_units, int n_rows, int n_heads, int head_dim, long keys,
                                        int* n_splits, int* n_waves) {
  const long c = keys;
  const long tiles = c < 1 ? 1 : (c + ATTN_DECODE_TILE_KEYS - 1) / ATTN_DECODE_TILE_KEYS;
  const long blocks = n_rows * n_heads < 1 ? 1 : (long)n_rows * n_heads;
  int nw = blocks > n_compute_units ? 4 : ATTN_DECODE_ROW_WAVES;
  const int fewest = head_dim > 128 ? 4 : 2;  // (the block's threads write a column of the head each)
  while (nw > fewest && nw / 2 >= tiles) nw /= 2;
  const long keys_a_wave = c / nw;
  long ns = 1;
  if (keys_a_wave >= ATTN_DECODE_SPLIT_KEYS_A_WAVE) {
    ns = keys_a_wave / ATTN_DECODE_KEYS_A_PART;
    if (n_compute_units / blocks < ns) ns = n_compute_units / blocks;
    if (ns > 64) ns = 64;
    if (ns < 1) ns = 1;
  }
  if (ns == 1 && blocks <= n_compute_units && c >= 2048) nw = 2 * ATTN_DECODE_ROW_WAVES;
  *n_splits = (int)ns, *n_waves = nw;
}
