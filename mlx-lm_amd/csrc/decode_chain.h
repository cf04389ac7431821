// All layers of a decode step of one or two rows as one launch (decode_chain.hip): what the host of a step
// gives it.  Layers are alike: LayerNorm, attention over pages, LayerNorm, tanh-GELU feed-forward, bfloat16.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#define CHAIN_MOST_ROWS 2
#define CHAIN_HEAD_DIM 64
#define CHAIN_MOST_KEYS 1024  // keys a row has in the cache before the step

// A layer's pointers; products: q/k/v, output projection, the feed-forward's two.
typedef struct {
  const void* W[4];  // packed: tiles of 16 features x 64 k
  const float* bias[4];
  const float* gamma[2];
  const float* beta[2];
  void* k_pages;
  void* v_pages;
} ChainLayer;

typedef struct {
  int n_layers, width, inner, n_heads, n_kv_heads, page_size;
  size_t page_stride;  // elements from a page's keys to the next page's
  float eps1, eps2, scale;
} ChainDims;

#ifdef __cplusplus
extern "C" {
#endif
// 1 if the launch takes these sizes
int decode_chain_takes(const ChainDims* d, int rows);
// bytes of the launch's own memory for this many rows; zeros before its first use, and used by one launch at a time
size_t decode_chain_bytes(const ChainDims* d, int rows);
// h_out = the stream `h` ([rows][width] float32, row stride ldh, both) after all layers; the rows' keys and values go to
// their pages.  `layers` lies on the device.  `blocks` and `patience` (ticks of 10 ns): 0, or for tests a smaller
// grid, and how long a block waits for another's unit before the units are dealt anew among the blocks that run.
int decode_chain(const ChainDims* d, int rows, const void* layers, void* memory, const float* h, float* h_out, int ldh,
                 const int* block_table, int max_blocks, const int* token_req, const int* positions, int blocks,
                 unsigned patience, hipStream_t stream);
#ifdef __cplusplus
}
#endif
