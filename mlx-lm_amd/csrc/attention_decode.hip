// Decode attention: one query row per block, keys streamed from the pages
// straight into registers (no LDS staging).  bfloat16 caches with head sizes
// 32, 64, 128 and 256, float caches with 16, 32, 64 and 128 (a lane holds 16 bytes of a
// key, and 4 to 32 lanes a key).  Same contract as attn_row in attention.hip
// (same arguments, same partial buffers, same merge); this is the kernel that
// serving uses, attn_row stays as the general one (any head size).
//
// Replaces scaled_dot_product_attention with one query per sequence
// (mlx_lm/models/base.py:132-139 with mask=None, mlx_lm/generate.py:1414).
//
// Work split: grid (rows, heads, n_splits), 1 to 16 waves a block.  The row's
// keys [k_lo, k_hi) are cut into tiles of 16 (of 32 where a load brings 16); the tiles are dealt to the splits
// in runs and, inside a block, to the waves in turn; a wave asks for its next tile before it takes one.  With few rows in a step
// it is the many waves of a block, joined through LDS, that give the GPU
// enough to do; the parts of splits are joined by the block of a (row, head) that
// finishes last, or by a second kernel.  A wave reads a tile as
// CPK-lane groups: lane l holds 16 bytes (EPL = 8 bfloat16 or 4 float columns)
// l % CPK of key l / CPK of each load, where CPK = head_dim / EPL lanes cover
// one key.  One load instruction therefore reads 64 / CPK whole keys that lie
// back to back in a page.  Scores: EPL products per lane, summed over the CPK
// lanes of the key by xor shuffles.  The weighted sum keeps, per lane, the EPL
// columns of *its* keys and is only joined over the lane groups (and then the
// waves) at the end.
#include "attention_decode_row.h"

// Where the parts of a (row, head) are counted that the kernel joins itself: all launches on a GPU share the counters, so launches that
// join and overlap on one GPU race.
#define JOIN_MAX_ITEMS 65536
static __device__ unsigned join_counters[JOIN_MAX_ITEMS];

// T: uint16_t (bfloat16 bits) or float.  CPK lanes per key: head_dim = EPL * CPK.  ONCE: every key is read by one block
// (as many key heads as query heads), with the streaming hint.  Where query heads share a key head, blocks that read the
// same keys find them in the die's L2 or on their way to it (which is why their rows are the fast index, below), and a hinted line
// is gone by then: 64 rows of 28 query heads
// of 128 over 4 key heads 819 us at contexts of 6,000 to 8,001 and 107 at 700 to 1,300, 691 and 79 without the hint; 32 of
// 32 over 8 396 and 294; float, 64 of 16 of 128 over 4 938 and 686.  (At few rows and short contexts it is the hint that is
// ahead there too, by 3 to 8 %: 8 rows of 16 of 64 over 4, 60 to 500 keys, 7.3 and 7.9 us.)
// SHAPED: scores also pass the soft cap and take the distance table's term.  A kernel of its own because a short walk waits
// for its instructions: the loop below holds the arithmetic four times, each with a tanh a load, and beside blocks that
// read weights ahead (2 rows of 25 heads of 64 at 60 to 500 keys) a launch took 9.3 us with them in and takes 8.9.
// Five waves a SIMD at most for bfloat16 heads of 64 with a key head each: without the tanh's registers seven fit, all blocks
// of 64 rows of 25 heads start at once and rows of unequal length end unevenly (a step of GPT-2 XL at 64 requests, contexts of
// 300 to 1,001, 4.74 ms with seven, 4.54 with five).  Heads that share keys are 1 to 6 % ahead with seven.
template <typename T, int CPK, bool ONCE, bool SHAPED>
__global__ __launch_bounds__(64 * (CPK >= 16 ? MAX_WAVES / 2 : MAX_WAVES))
__attribute__((amdgpu_waves_per_eu(CPK >= 16 ? 2 : 4, CPK == 8 && sizeof(T) == 2 && ONCE ? 5 : 8))) void attn_decode_kernel(DecodeArgs p) {
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), n_waves = blockDim.x >> 6;
  if (blockIdx.y >= p.n_heads) {  // a reading block (uniform)
    if (blockIdx.z != 0) return;
    // blocks go to the dies in turn, in the order x, y, z: this one is on die `lin % 8`, and
    // block j of the product to come, which reads chunk j, on die j % 8
    const int r = blockIdx.x + gridDim.x * (blockIdx.y - p.n_heads);
    const int readers = gridDim.x * (gridDim.y - p.n_heads);
    const int lin = gridDim.x * p.n_heads + r;
    const int die = lin & 7, rank = r >> 3, per_die = (readers + 7) >> 3;
    // the die's chunks (die, die + 8, ...) laid end to end and cut into equal shares, one a block
    const size_t mine = die < p.ahead_chunks ? (size_t)((p.ahead_chunks - die + 7) / 8) * p.ahead_pieces : 0;
    const size_t share = (mine + per_die - 1) / per_die;
    const size_t lo = (size_t)rank * share, hi = min(lo + share, mine);
    unsigned int seen = 0u;
    for (size_t i0 = lo + tid; i0 < hi; i0 += 8 * (size_t)blockDim.x) {
      uint4 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const size_t t = min(i0 + u * (size_t)blockDim.x, hi - 1);
        const size_t c = t / p.ahead_pieces;
        v[u] = p.ahead[((size_t)die + 8 * c) * p.ahead_pieces + (t - c * p.ahead_pieces)];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) seen |= v[u].x;
    }
    asm volatile("" ::"v"(seen));  // the loads stay although nobody wants the values
    return;
  }
  // With a key head each, a row's heads are neighbours in the launch.  Blocks go to the compute units in turn, so with the rows as
  // the fast index and 64 rows every 256th block was the same row's: a unit had the longest row's heads and no others.  25 heads of
  // 64, us, rows fast and heads fast: 64 rows at 300 to 1,001 keys 47.7 and 46.7, 48 at 16 to 1,000 32.3 and 30.5, 16 at 500 to
  // 8,001 100 and 90, 8 at 4,000 to 8,001 57.9 and 56.5; rows of one length, 24 of 550 and 8 of 6,000, 18.0 and 18.0, 48.3 and 49.
  // Where heads share keys the rows are the fast index: blocks go to the eight dies in turn too, and at a multiple of eight rows the
  // heads of a group are on one die, whose L2 has the keys after the first.  As neighbours they are on as many dies, each of
  // which reads the keys; rows fast and heads fast: 32 heads of 128 over 8, 8 rows at 60 to 500 keys 9.9 and 12.3, at 4,000 to
  // 8,001 83.5 and 126, 12 at 500 to 3,000 57.6 and 60.0, 64 at 300 to 1,001 71.3 and 108, at 2,000 to 6,000 397 and 628; 28 over 4,
  // the same, 10.0 / 11.5, 83 / 107, 57 / 62, 58 / 92, 388 / 553; float, 24 of 128 over 8, 64 at 300 to 1,001 110 and 161.
  int item = blockIdx.x, h = blockIdx.y;
  if constexpr (ONCE) {
    const int lin = blockIdx.x + gridDim.x * blockIdx.y;
    item = lin / p.n_heads, h = lin - item * p.n_heads;
  }
  attend_row<T, CPK, ONCE, SHAPED, MAX_WAVES, true>(p, wave, n_waves, item, h, blockIdx.z, join_counters);
}

// attn_decode_group: bfloat16, the query heads that share a key head taken together.  Where many
// query heads read one key head (a latent that all heads share, large groups), a block a (row,
// head) walks the same keys once a head and pays a key's instructions each time.  Here a block
// takes a (row, key head, sixteen of its query heads, part of the keys), a wave sixteen keys at a
// time, on the matrix cores:
//   S^T = K Q^T   v_mfma_f32_16x16x32_bf16: keys are the rows (lane l brings 16 bytes of key l % 16
//                 straight from its page), the heads the columns (the queries stay in registers);
//                 a lane then holds four keys' scores of head l % 16.
//   O^T += V^T P^T  v_mfma_f32_16x16x16_bf16: those four weights are the lane's fragment of P^T as
//                 they are; the lane brings column 16 d + l % 16 of its four keys' values.
// Online softmax per head in 32-bit; the waves' results are joined through LDS in the waves'
// order, the parts of a split row by attn_decode_merge_kernel.
typedef __attribute__((ext_vector_type(4))) short s16x4_t;

template <int HD>
__global__ __launch_bounds__(256) void attn_decode_group_kernel(DecodeArgs p, int group, int head_tiles) {
  constexpr int QC = HD / 32;      // steps of K Q^T
  constexpr int DT = HD / 16;      // 16-row tiles of O^T
  constexpr int OS = HD + 1;       // a head's row in Os (the odd stride keeps sixteen heads on sixteen banks)
  __shared__ float Ms[4][16], Ls[4][16];
  extern __shared__ int group_lds[];
  float* Os = (float*)group_lds;                 // [4 waves][16 heads][OS]
  int* pages = group_lds + 4 * 16 * OS;          // [max_blocks] with table_in_lds
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, c16 = lane & 15;
  const int item = blockIdx.x, split = blockIdx.z;
  const int kv_head = blockIdx.y / head_tiles, ht = blockIdx.y % head_tiles;
  const int row = p.rows_are_requests ? item : p.rows[item];
  const int req = p.rows_are_requests ? item : p.token_req[row];
  const int* table = p.block_table + (size_t)req * p.max_blocks;
  if (p.table_in_lds)
    for (int i = tid; i < p.max_blocks; i += 256) pages[i] = table[i];
  const int pos = p.positions[row];
  const uint16_t* k_pages = (const uint16_t*)p.k_pages;
  const uint16_t* v_pages = (const uint16_t*)p.v_pages;
  const int in_group = ht * 16 + c16;  // this lane's head within the group
  const int head = kv_head * group + min(in_group, group - 1);
  Frag8g qf[QC];
  {
    const uint16_t* qrow = (const uint16_t*)p.q + (size_t)row * p.ldq + (size_t)head * HD + 8 * g;
#pragma unroll
    for (int c = 0; c < QC; ++c) {
      qf[c].u = *(const uint4*)(qrow + 32 * c);
      if (in_group >= group) qf[c].u = make_uint4(0u, 0u, 0u, 0u);
    }
  }
  const int k_hi = pos + 1;
  const int k_lo = p.window > 0 ? max(0, pos - p.window + 1) : 0;
  const int kt0 = (k_lo / 16) * 16;
  const int n_tiles = (k_hi - kt0 + 15) / 16;
  const int per_split = (n_tiles + p.n_splits - 1) / p.n_splits;
  const int t_begin = split * per_split, t_end = min(n_tiles, t_begin + per_split);
  float m = -INFINITY, l = 0.f;
  f32x4_t o[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) o[d] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const size_t head_off = (size_t)kv_head * p.page_size * HD;
  if (p.table_in_lds) __syncthreads();  // (uniform over the block)
  auto page_of_key = [&](int key) { return p.table_in_lds ? pages[key / p.page_size] : table[key / p.page_size]; };

  for (int t = t_begin + wave; t < t_end; t += 4) {
    const int kt = kt0 + t * 16;
    Frag8g kf[QC];
    {
      const int key = min(max(kt + c16, k_lo), k_hi - 1);  // (keys outside the run: pulled inside, masked below)
      const uint16_t* kp = k_pages + (size_t)page_of_key(key) * p.page_stride + head_off + (size_t)(key % p.page_size) * HD + 8 * g;
#pragma unroll
      for (int c = 0; c < QC; ++c) kf[c].u = *(const uint4*)(kp + 32 * c);
    }
    const uint16_t* vp[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int key = min(max(kt + 4 * g + x, k_lo), k_hi - 1);
      vp[x] = v_pages + (size_t)page_of_key(key) * p.page_stride + head_off + (size_t)(key % p.page_size) * HD + c16;
    }
    s16x4_t va[DT];
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int x = 0; x < 4; ++x) va[d][x] = (short)vp[x][16 * d];
    f32x4_t s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < QC; ++c) s = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[c].v, qf[c].v, s, 0, 0, 0);
    float sx[4], tmax = -INFINITY;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int key = kt + 4 * g + x;
      sx[x] = (key >= k_lo && key < k_hi) ? s[x] * p.scale : -INFINITY;
      tmax = fmaxf(tmax, sx[x]);
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16, WAVE));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, WAVE));
    const float m_new = fmaxf(m, tmax);  // finite: every tile holds at least one live key
    const float alpha = __expf(m - m_new);
    s16x4_t pb;
    float psum = 0.f;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const float px = __expf(sx[x] - m_new);  // exp(-inf) = 0 for masked keys
      psum += px;
      pb[x] = (short)f32_to_bf16_bits(px);
    }
    l = l * alpha + psum;
#pragma unroll
    for (int d = 0; d < DT; ++d) {
#pragma unroll
      for (int x = 0; x < 4; ++x) o[d][x] *= alpha;
      o[d] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(va[d], pb, o[d], 0, 0, 0);
    }
    m = m_new;
  }
  // the four lane groups of a head hold sums over different keys
  l += __shfl_xor(l, 16, WAVE);
  l += __shfl_xor(l, 32, WAVE);
  if (g == 0) Ms[wave][c16] = m, Ls[wave][c16] = l;
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int x = 0; x < 4; ++x) Os[((size_t)wave * 16 + c16) * OS + 16 * d + 4 * g + x] = o[d][x];
  __syncthreads();
  for (int e = tid; e < 16 * HD; e += 256) {
    const int hh = e / HD, col = e - hh * HD;
    if (ht * 16 + hh >= group) continue;
    float M = -INFINITY;
    for (int w = 0; w < 4; ++w) M = fmaxf(M, Ms[w][hh]);
    float L = 0.f, acc = 0.f;
    for (int w = 0; w < 4; ++w) {
      const float f = (Ms[w][hh] == -INFINITY) ? 0.f : __expf(Ms[w][hh] - M);
      L += Ls[w][hh] * f;
      acc += Os[((size_t)w * 16 + hh) * OS + col] * f;
    }
    const int hq = kv_head * group + ht * 16 + hh;
    if (p.n_splits == 1) {
      put((uint16_t*)p.out + out_at(p, row, hq * HD + col), acc / with_sink(p, hq, M, L) * head_gate_of(p, row, hq));
    } else {
      const size_t base = ((size_t)item * p.n_heads + hq) * p.n_splits + split;
      p.part_o[base * HD + col] = acc;
      if (col == 0) p.part_ml[base * 2] = M, p.part_ml[base * 2 + 1] = L;
    }
  }
}

// grid (rows, heads), HD threads: join the splits
template <typename T, int CPK>
__global__ void attn_decode_merge_kernel(DecodeArgs p) {
  constexpr int HD = 16 / sizeof(T) * CPK;
  const int item = blockIdx.x, h = blockIdx.y, d = threadIdx.x;
  const int row = p.rows_are_requests ? item : p.rows[item];
  const size_t base = ((size_t)item * p.n_heads + h) * p.n_splits;
  float M = -INFINITY;
  for (int s = 0; s < p.n_splits; ++s) M = fmaxf(M, p.part_ml[(base + s) * 2]);
  float L = 0.f, acc = 0.f;
  for (int s = 0; s < p.n_splits; ++s) {
    const float ms = p.part_ml[(base + s) * 2];
    if (ms == -INFINITY) continue;
    const float w = __expf(ms - M);
    L += p.part_ml[(base + s) * 2 + 1] * w;
    acc += p.part_o[(base + s) * HD + d] * w;
  }
  put((T*)p.out + out_at(p, row, h * HD + d), acc / with_sink(p, h, M, L) * head_gate_of(p, row, h) * gate_at<T>(p, row, h * HD + d));
}

DEFINE_LAST_ERROR(mlxlm_last_error)

template <typename T, int CPK>
static void launch(const DecodeArgs& p, int n_rows, int n_waves, hipStream_t stream) {
  // reading blocks for the CUs that the rows leave idle, if there are eight or more
  int extra_y = 0;
  if (p.ahead && p.ahead_chunks > 0) {
    extra_y = (n_compute_units() - n_rows * p.n_heads * p.n_splits) / n_rows;
    if (extra_y * n_rows < 8) extra_y = 0;
  }
  const size_t lds = p.table_in_lds ? (size_t)p.max_blocks * sizeof(int) : 0;
  const dim3 grid(n_rows, p.n_heads + extra_y, p.n_splits), block(64 * n_waves);
  const bool once = p.n_heads == p.n_kv_heads, shaped = p.softcap > 0.f || p.dist_bias;
  if (once && !shaped)
    hipLaunchKernelGGL((attn_decode_kernel<T, CPK, true, false>), grid, block, lds, stream, p);
  else if (!shaped)
    hipLaunchKernelGGL((attn_decode_kernel<T, CPK, false, false>), grid, block, lds, stream, p);
  else if (once)
    hipLaunchKernelGGL((attn_decode_kernel<T, CPK, true, true>), grid, block, lds, stream, p);
  else
    hipLaunchKernelGGL((attn_decode_kernel<T, CPK, false, true>), grid, block, lds, stream, p);
  if (p.n_splits > 1 && !p.join_here)
    hipLaunchKernelGGL((attn_decode_merge_kernel<T, CPK>), dim3(n_rows, p.n_heads), dim3(16 / sizeof(T) * CPK), 0, stream, p);
}

// Same arguments as attn_row, with what is read ahead and rows_are_requests between: 1 says that
// item i of `rows` is row i and belongs to request i (every request of the step brings one token),
// which saves the kernel two trips to memory.  dtype DT_BF16 with head_dim 32, 64, 128 or 256, DT_F32
// with 16, 32, 64 or 128, and pages that hold whole loads (page_size a multiple of the keys in 1 KB).
// join_in_kernel: 0, a second kernel joins the n_splits parts of a (row, head); 1, the block that
// finishes a (row, head) last does (up to 65,536 (row, head)s; part_o and part_ml are still where
// the parts pass through); 2, the same, and n_splits is only the most a row takes: a short row
// takes fewer, by its own length.
// Launches that join in the kernel and overlap on one GPU race (they share the counters).
static int decode_rows_launch(void* out, const void* q, int ldq, int ldo, const void* k_pages,
                              const void* v_pages, size_t page_stride, const int* block_table,
                              int max_blocks, const int* token_req, const int* positions,
                              const int* rows, int n_rows, int n_heads, int n_kv_heads, int head_dim,
                              int page_size, int window, float scale, int n_splits, float* part_o,
                              float* part_ml, int n_waves, const void* ahead, size_t ahead_chunk_bytes,
                              int ahead_chunks, int rows_are_requests, int dtype, int join_in_kernel,
                              const float* head_scale, const float* slopes,
                              const void* gate, int ldg, int keep_first, const AttnTerms* shape, hipStream_t stream) {
  if (n_rows <= 0) return 0;
  if (shape && (shape->softcap < 0.f || (shape->dist_bias && shape->n_dist <= 0)))
    FAIL("attn_decode: softcap %g, a distance table of %d entries a head", (double)shape->softcap, shape->n_dist);
  if (keep_first < 0) FAIL("attn_decode: keep_first %d must not be negative", keep_first);
  if (gate && ldg < n_heads * head_dim) FAIL("attn_decode: the gate's row stride %d is smaller than its rows", ldg);
  if (dtype != DT_F32 && dtype != DT_BF16) FAIL("attn_decode: unknown dtype code %d", dtype);
  const int epl = dtype == DT_F32 ? 4 : 8;  // elements in a lane's 16 bytes
  if (n_waves < 1 || n_waves > MAX_WAVES) FAIL("attn_decode: %d waves a block, must be 1 to %d", n_waves, MAX_WAVES);
  if (head_dim != 4 * epl && head_dim != 8 * epl && head_dim != 16 * epl && head_dim != 32 * epl)
    FAIL("attn_decode: head_dim %d is not %d, %d, %d or %d (attn_row takes the others)", head_dim, 4 * epl, 8 * epl,
         16 * epl, 32 * epl);
  const int cpk = head_dim / epl;
  if (head_dim > 64 * n_waves) FAIL("attn_decode: head_dim %d needs at least %d waves", head_dim, (head_dim + 63) / 64);
  if (cpk >= 16 && n_waves > MAX_WAVES / 2) n_waves = MAX_WAVES / 2;  // (those kernels' registers allow eight)
  const int kpl = 64 / cpk;
  if (page_size <= 0 || page_size % kpl != 0)
    FAIL("attn_decode: page_size %d must be a multiple of %d for head_dim %d", page_size, kpl, head_dim);
  if (n_heads <= 0 || n_kv_heads <= 0 || n_heads % n_kv_heads != 0)
    FAIL("attn_decode: %d query heads cannot be grouped over %d key heads", n_heads, n_kv_heads);
  if (!out || !q || !k_pages || !v_pages || !block_table || !token_req || !positions || !rows)
    FAIL("attn_decode: null pointer");
  if (ldq % epl != 0 || ((uintptr_t)q & 15)) FAIL("attn_decode: queries must be 16-byte aligned rows");
  if (page_stride % epl != 0 || (((uintptr_t)k_pages | (uintptr_t)v_pages) & 15))
    FAIL("attn_decode: pages must be 16-byte aligned");
  if (window < 0) FAIL("attn_decode: window %d must not be negative", window);
  if (n_splits < 1 || n_splits > 65535) FAIL("attn_decode: n_splits %d out of range", n_splits);
  if (n_splits > 1 && (!part_o || !part_ml)) FAIL("attn_decode: splits need the partial buffers");
  DecodeArgs p;
  p.out = out, p.q = q, p.k_pages = k_pages, p.v_pages = v_pages;
  p.block_table = block_table, p.token_req = token_req, p.positions = positions, p.rows = rows;
  p.part_o = part_o, p.part_ml = part_ml, p.page_stride = page_stride;
  p.ldq = ldq, p.ldo = ldo, p.max_blocks = max_blocks;
  p.n_heads = n_heads, p.n_kv_heads = n_kv_heads, p.page_size = page_size;
  p.window = window, p.n_splits = n_splits, p.scale = scale;
  p.head_scale = head_scale, p.slopes = slopes, p.gate = gate, p.ldg = ldg;
  p.keep_first = window > 0 ? keep_first : 0;
  p.softcap = shape ? shape->softcap : 0.f, p.dist_bias = shape ? shape->dist_bias : nullptr;
  p.n_dist = shape ? shape->n_dist : 0;
  p.sinks = shape ? shape->sinks : nullptr, p.head_gate = shape ? shape->head_gate : nullptr;
  p.ldhg = shape ? shape->ldhg : 0;
  if (p.head_gate && p.ldhg < n_heads) FAIL("attn_decode: the heads' gate has rows of %d columns", p.ldhg);
  if (ahead && (((uintptr_t)ahead & 15) || ahead_chunk_bytes % 16 != 0 || ahead_chunks < 0))
    FAIL("attn_decode: what is read ahead must be chunks of 16-byte pieces");
  p.ahead = (const uint4*)ahead, p.ahead_pieces = ahead ? ahead_chunk_bytes / 16 : 0;
  p.ahead_chunks = ahead ? ahead_chunks : 0;
  p.out_head_dim = head_dim;
  if (ldo == 0 && dtype != DT_BF16) FAIL("attn_decode: the packed order (ldo == 0) is for a bfloat16 out");
  p.rows_are_requests = rows_are_requests ? 1 : 0;
  // (more (row, head)s than counters: the second kernel joins the parts)
  if (join_in_kernel < 0 || join_in_kernel > 2) FAIL("attn_decode: join_in_kernel %d is not 0, 1 or 2", join_in_kernel);
  p.join_here = n_splits > 1 && (long)n_rows * n_heads <= JOIN_MAX_ITEMS ? join_in_kernel : 0;
  p.table_in_lds = max_blocks > 0 && max_blocks <= 8192;  // (32 KB of LDS at most)
  p.page_shift = (page_size & (page_size - 1)) == 0 ? __builtin_ctz(page_size) : -1;
  if (dtype == DT_BF16) {
    if (cpk == 4)
      launch<uint16_t, 4>(p, n_rows, n_waves, stream);
    else if (cpk == 8)
      launch<uint16_t, 8>(p, n_rows, n_waves, stream);
    else if (cpk == 16)
      launch<uint16_t, 16>(p, n_rows, n_waves, stream);
    else
      launch<uint16_t, 32>(p, n_rows, n_waves, stream);
  } else {
    if (cpk == 4)
      launch<float, 4>(p, n_rows, n_waves, stream);
    else if (cpk == 8)
      launch<float, 8>(p, n_rows, n_waves, stream);
    else if (cpk == 16)
      launch<float, 16>(p, n_rows, n_waves, stream);
    else
      launch<float, 32>(p, n_rows, n_waves, stream);
  }
  CHECK_LAUNCH("attn_decode");
  return 0;
}

// attn_decode_rows_biased: with the optional terms of DecodeArgs (null or 0 where one is absent).
extern "C" int attn_decode_rows_biased(void* out, const void* q, int ldq, int ldo, const void* k_pages,
                                       const void* v_pages, size_t page_stride, const int* block_table,
                                       int max_blocks, const int* token_req, const int* positions,
                                       const int* rows, int n_rows, int n_heads, int n_kv_heads, int head_dim,
                                       int page_size, int window, float scale, int n_splits, float* part_o,
                                       float* part_ml, int n_waves, const void* ahead, size_t ahead_chunk_bytes,
                                       int ahead_chunks, int rows_are_requests, int dtype,
                                       int join_in_kernel, const float* head_scale, const float* slopes,
                                       const void* gate, int ldg, int keep_first, hipStream_t stream) {
  return decode_rows_launch(out, q, ldq, ldo, k_pages, v_pages, page_stride, block_table, max_blocks, token_req,
                            positions, rows, n_rows, n_heads, n_kv_heads, head_dim, page_size, window, scale,
                            n_splits, part_o, part_ml, n_waves, ahead, ahead_chunk_bytes, ahead_chunks,
                            rows_are_requests, dtype, join_in_kernel, head_scale, slopes, gate, ldg,
                            keep_first, nullptr, stream);
}

// attn_decode_rows_terms: every optional term, as an AttnTerms (attention_tiles.h); null: none.
extern "C" int attn_decode_rows_terms(void* out, const void* q, int ldq, int ldo, const void* k_pages,
                                      const void* v_pages, size_t page_stride, const int* block_table,
                                      int max_blocks, const int* token_req, const int* positions,
                                      const int* rows, int n_rows, int n_heads, int n_kv_heads, int head_dim,
                                      int page_size, int window, float scale, int n_splits, float* part_o,
                                      float* part_ml, int n_waves, const void* ahead, size_t ahead_chunk_bytes,
                                      int ahead_chunks, int rows_are_requests, int dtype,
                                      int join_in_kernel, const AttnTerms* t, hipStream_t stream) {
  return decode_rows_launch(out, q, ldq, ldo, k_pages, v_pages, page_stride, block_table, max_blocks, token_req,
                            positions, rows, n_rows, n_heads, n_kv_heads, head_dim, page_size, window, scale,
                            n_splits, part_o, part_ml, n_waves, ahead, ahead_chunk_bytes, ahead_chunks,
                            rows_are_requests, dtype, join_in_kernel, t ? t->head_scale : nullptr,
                            t ? t->slopes : nullptr, t ? t->gate : nullptr, t ? t->ldg : 0, t ? t->keep_first : 0, t,
                            stream);
}

extern "C" int attn_decode_rows(void* out, const void* q, int ldq, int ldo, const void* k_pages,
                                const void* v_pages, size_t page_stride, const int* block_table,
                                int max_blocks, const int* token_req, const int* positions,
                                const int* rows, int n_rows, int n_heads, int n_kv_heads, int head_dim,
                                int page_size, int window, float scale, int n_splits, float* part_o,
                                float* part_ml, int n_waves, const void* ahead, size_t ahead_chunk_bytes,
                                int ahead_chunks, int rows_are_requests, int dtype,
                                int join_in_kernel, hipStream_t stream) {
  return attn_decode_rows_biased(out, q, ldq, ldo, k_pages, v_pages, page_stride, block_table, max_blocks, token_req,
                                 positions, rows, n_rows, n_heads, n_kv_heads, head_dim, page_size, window, scale,
                                 n_splits, part_o, part_ml, n_waves, ahead, ahead_chunk_bytes, ahead_chunks,
                                 rows_are_requests, dtype, join_in_kernel, nullptr, nullptr, nullptr, 0, 0,
                                 stream);
}

// attn_decode_group: the rows of attn_decode_rows for bfloat16 caches with head_dim 64, 128 or 256,
// all query heads of a key head in one block (see attn_decode_group_kernel).  n_splits parts of a
// row's keys (part_o: n_rows * n_heads * n_splits * head_dim floats, part_ml: two a part; joined
// by a second kernel).  ldo == 0: out in the packed order.  t: of the optional terms the sinks and the
// heads' gate, or null.
extern "C" int attn_decode_group(void* out, const void* q, int ldq, int ldo, const void* k_pages, const void* v_pages,
                                 size_t page_stride, const int* block_table, int max_blocks, const int* token_req,
                                 const int* positions, const int* rows, int n_rows, int n_heads, int n_kv_heads,
                                 int head_dim, int page_size, int window, float scale, int n_splits, float* part_o,
                                 float* part_ml, int rows_are_requests, const AttnTerms* t, hipStream_t stream) {
  if (n_rows <= 0) return 0;
  if (head_dim != 64 && head_dim != 128 && head_dim != 256) FAIL("attn_decode_group: head_dim %d is not 64, 128 or 256", head_dim);
  if (n_heads <= 0 || n_kv_heads <= 0 || n_heads % n_kv_heads != 0)
    FAIL("attn_decode_group: %d query heads cannot be grouped over %d key heads", n_heads, n_kv_heads);
  if (!out || !q || !k_pages || !v_pages || !block_table || !token_req || !positions || !rows)
    FAIL("attn_decode_group: null pointer");
  if (page_size <= 0 || window < 0) FAIL("attn_decode_group: page_size %d, window %d", page_size, window);
  if (ldq % 8 != 0 || ((uintptr_t)q & 15)) FAIL("attn_decode_group: queries must be 16-byte aligned rows");
  if (page_stride % 8 != 0 || (((uintptr_t)k_pages | (uintptr_t)v_pages) & 15))
    FAIL("attn_decode_group: pages must be 16-byte aligned");
  if (n_splits < 1 || n_splits > 65535) FAIL("attn_decode_group: %d parts", n_splits);
  if (n_splits > 1 && (!part_o || !part_ml)) FAIL("attn_decode_group: parts need part_o and part_ml");
  DecodeArgs p = {};
  p.out = out, p.q = q, p.k_pages = k_pages, p.v_pages = v_pages;
  p.block_table = block_table, p.token_req = token_req, p.positions = positions, p.rows = rows;
  p.part_o = part_o, p.part_ml = part_ml, p.page_stride = page_stride;
  p.ldq = ldq, p.ldo = ldo, p.max_blocks = max_blocks;
  p.n_heads = n_heads, p.n_kv_heads = n_kv_heads, p.page_size = page_size, p.window = window, p.n_splits = n_splits;
  p.scale = scale, p.out_head_dim = head_dim, p.rows_are_requests = rows_are_requests ? 1 : 0;
  p.table_in_lds = max_blocks > 0 && max_blocks <= 8192;
  if (t) {
    if (t->head_scale || t->slopes || t->gate || t->keep_first > 0 || t->softcap > 0.f || t->dist_bias)
      FAIL("attn_decode_group: of the optional terms only sinks and the heads' gate");
    if (t->head_gate && t->ldhg < n_heads) FAIL("attn_decode_group: the heads' gate has rows of %d columns", t->ldhg);
    p.sinks = t->sinks, p.head_gate = t->head_gate, p.ldhg = t->ldhg;
  }
  const int group = n_heads / n_kv_heads, head_tiles = (group + 15) / 16;
  if ((long)n_kv_heads * head_tiles > 65535) FAIL("attn_decode_group: %d key heads in a launch", n_kv_heads);
  const size_t lds = (size_t)4 * 16 * (head_dim + 1) * sizeof(float) + (p.table_in_lds ? (size_t)max_blocks * sizeof(int) : 0);
  const dim3 grid(n_rows, n_kv_heads * head_tiles, n_splits), block(256);
#define LAUNCH_GROUP(HD)                                                                                             \
  do {                                                                                                               \
    static bool raised = false;                                                                                      \
    if (!raised) {                                                                                                   \
      (void)hipFuncSetAttribute((const void*)attn_decode_group_kernel<HD>, hipFuncAttributeMaxDynamicSharedMemorySize, \
                                120 * 1024);                                                                         \
      raised = true;                                                                                                 \
    }                                                                                                                \
    hipLaunchKernelGGL((attn_decode_group_kernel<HD>), grid, block, lds, stream, p, group, head_tiles);              \
    if (n_splits > 1)                                                                                                \
      hipLaunchKernelGGL((attn_decode_merge_kernel<uint16_t, HD / 8>), dim3(n_rows, n_heads), dim3(HD), 0, stream, p); \
  } while (0)
  if (head_dim == 64)
    LAUNCH_GROUP(64);
  else if (head_dim == 128)
    LAUNCH_GROUP(128);
  else
    LAUNCH_GROUP(256);
#undef LAUNCH_GROUP
  CHECK_LAUNCH("attn_decode_group");
  return 0;
}
