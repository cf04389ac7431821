// Linear layer on bfloat16 operands with MFMA and 32-bit accumulation:
//   out[m, n] = epilogue( sum_k A[m, k] * W[n, k] + bias[n] )
// A is [M, K] activations, W is [N, K] (the [out, in] layout of a linear
// layer), both contiguous along k, which is what both MFMA operands want.
// Epilogues: plain, tanh-GELU, or accumulate into a 32-bit residual stream.
// Replaces nn.Linear calls of the reference (mlx_lm/models/gpt2.py:41-42,52,
// 68,76-80) and the tied head (mlx_lm/models/gpt2.py:167).
//
// Two kernels:
//  * gemm_bf16_tile: block tiles of 32 x 128 to 256 x 256 outputs, k-blocks of 64 columns
//    copied from memory straight into a ring in LDS, several ahead; waves of 32 x 32
//    v_mfma_f32_32x32x16_bf16 tiles; each die gets a run of neighbouring tiles that share
//    their operands in its L2; K may be split over blocks where rows are few.  Any M, N; K % 8 == 0.
//  * gemm_bf16_skinny: M <= 64 rows (decode).  A block of four waves owns 16
//    output features and splits K among its waves; W streams from HBM once
//    as the MFMA A-operand, the activations are the B-operand.
#include "common.h"
#include "lds_copy.h"
#include "tile_order.h"

#include <type_traits>

#define FLAG_GELU FLAG_ACT_GELU
#define FLAG_RELU2 FLAG_ACT_RELU2  // the square of the ReLU instead
#define FLAG_ACCUMULATE 2
#define FLAG_OUT_F32 4
#define FLAG_KV 8  // columns from q_width on are keys, then values: they go to their cache pages, not to out
#define FLAG_THROUGH 16  // (set here) out and ws are below 4 GB: the tile kernels' stores go through to memory

// Out-of-range loads (of the kernel for few rows) read a clamped address and are zeroed afterwards
// with this constant: selecting between an address and a zero kept in a variable turns the load
// into a flat load through scratch memory.
#define ZERO4 make_uint4(0u, 0u, 0u, 0u)

struct GemmArgs {
  const uint16_t* A;
  const uint16_t* W;
  const float* bias;
  void* out;
  int M, N, K;
  int lda, ldw, ldo;
  int flags;
  // K split over blockIdx.y (tiles 128 columns wide): partial sums [n_splits][M][N] go to ws
  float* ws;
  int n_splits, blocks_per_split;
  // key/value scatter (FLAG_KV): row m is token m of the step, at positions[m] of request token_req[m]
  uint16_t* k_pages;
  uint16_t* v_pages;
  size_t page_stride;
  const int* block_table;
  const int* token_req;
  const int* positions;
  int max_blocks, q_width, kv_width, head_dim, page_size;
  // W in the decode kernels' packed order instead of row-major (ldw == 0 at the entry point):
  // tiles of 16 features x 64 k (1024 elements), zero padded, w_kblocks of them a feature block;
  // in a tile the 8 values k = 16 g + 8 h + 0..7 of feature f lie at ((4 h + g) * 16 + f) * 8.
  int w_packed, w_kblocks;
  int tile_blocks;  // blocks of the grid's first dimension that have tiles: those behind them read weights ahead (read_weights)
};

// Element offset of the 16-byte piece `piece` (k = 8 piece ..) of feature row n in k-block 0.
__device__ __forceinline__ int packed_piece(int n, int piece, int w_kblocks) {
  return (n >> 4) * w_kblocks * 1024 + ((((piece & 1) << 2) + (piece >> 1)) * 16 + (n & 15)) * 8;
}

// Where column n (a key's or a value's: n >= q_width) of token m lies in the cache pages.
__device__ __forceinline__ uint16_t* kv_place(const GemmArgs& p, int m, int n) {
  const int c = n - p.q_width;
  const bool is_v = c >= p.kv_width;
  const int cc = is_v ? c - p.kv_width : c;
  const int head = cc / p.head_dim, d = cc - head * p.head_dim;
  const int pos = p.positions[m];
  const int page = p.block_table[(size_t)p.token_req[m] * p.max_blocks + pos / p.page_size];
  return (is_v ? p.v_pages : p.k_pages) + (size_t)page * p.page_stride +
         ((size_t)head * p.page_size + pos % p.page_size) * p.head_dim + d;
}

__device__ __forceinline__ void store_out(const GemmArgs& p, int m, int n, float v) {
  if (p.bias) v += p.bias[n];
  v = activate<true>(p.flags, v);
  if ((p.flags & FLAG_KV) && n >= p.q_width) {
    *kv_place(p, m, n) = f32_to_bf16_bits(v);
    return;
  }
  const size_t idx = (size_t)m * p.ldo + n;
  if (p.flags & FLAG_ACCUMULATE) {
    float* o = (float*)p.out;
    o[idx] += v;
  } else if (p.flags & FLAG_OUT_F32) {
    ((float*)p.out)[idx] = v;
  } else {
    ((uint16_t*)p.out)[idx] = f32_to_bf16_bits(v);
  }
}

// ---------------------------------------------------------------------------

#define BK 64

// The shape of a block: WAVES_M x WAVES_N waves, each with TM x TN MFMA tiles of 32 x 32, and rings in LDS of SLOTS_A
// k-blocks of the rows and SLOTS_B of the weights.  What bounds this kernel is how fast a CU is fed from the L2s (some 32 to 39 bytes a cycle arrive, measured with
// the products taken out), so the larger the tile, the fewer bytes per product: 256 x 256 where the matrix gives a tile
// to every CU, smaller ones where it does not; `price` below chooses.  Eight waves (but for 32 rows): two a SIMD cover each
// other's waits for LDS; four waves of 64 x 64 were level or up to 12 % behind.
// COPIERS: waves beside those that only copy (Tile128Fed).
// The widest shapes have room for two k-blocks of both and what is left goes to the weights, which come from memory while
// the rows lie in the L2s; their copies are asked for a few at a time between products (SPREAD): a wave that asks waits
// until its copies are taken, 64 KB a k-block, and right behind the barrier all waves did so at once, the matrix units idle.  Zeros, so that
// power does not limit, 256 x 256, a k-block: products alone 0.87 us, copies alone 0.96, both 1.28 and now 1.10; from memory, rows x features x K:
// 2,048 x 4,800 x 1,600 37.4 -> 33.6 us, x 6,400 x 1,600 47.4 -> 43.8, 8,000 x 4,800 x 1,600 128.3 -> 124, 8,000 x 1,280 x 5,120 111 -> 104.  The
// smaller shapes were level or up to 3 % slower with either (128 x 128 with five slots, 64 x 128 with six: what they wait for is not depth).
template <int WAVES_M_, int WAVES_N_, int TM_, int TN_, int SLOTS_A_, int PANEL_, int WAVES_PER_SIMD_, int SLOTS_B_ = SLOTS_A_, bool SPREAD_ = false, int COPIERS_ = 0>
struct TileShape {
  static constexpr int COPIERS = COPIERS_;
  static constexpr int WAVES_M = WAVES_M_, WAVES_N = WAVES_N_, TM = TM_, TN = TN_, SLOTS_A = SLOTS_A_, SLOTS_B = SLOTS_B_;
  static constexpr bool SPREAD = SPREAD_;
  static constexpr int PANEL = PANEL_, WAVES_PER_SIMD = WAVES_PER_SIMD_;  // PANEL: rows of tiles that share a die's L2
  static constexpr int WAVES = WAVES_M * WAVES_N, THREADS = 64 * (WAVES + COPIERS), ASKERS = COPIERS ? COPIERS : WAVES;
  static constexpr int BM = WAVES_M * TM * 32, BN = WAVES_N * TN * 32;
  static constexpr int PA = BM / 8 / ASKERS, PB = BN / 8 / ASKERS;  // copies of 1 KB a wave asks for per k-block
  static constexpr int COPIES = PA + PB;
  static constexpr int A_BYTES = BM * BK * 2, B_BYTES = BN * BK * 2, RING = SLOTS_A * A_BYTES + SLOTS_B * B_BYTES;
  // as many slots for both: a k-block's rows and weights side by side, one address for both; else a ring behind the other
  static constexpr bool ALIKE = SLOTS_A == SLOTS_B;
  static constexpr int A_STRIDE = ALIKE ? A_BYTES + B_BYTES : A_BYTES, B_STRIDE = ALIKE ? A_STRIDE : B_BYTES;
  static constexpr int B_BASE = ALIKE ? A_BYTES : SLOTS_A * A_BYTES;
  static_assert(BM % (8 * ASKERS) == 0 && BN % (8 * ASKERS) == 0, "a wave copies whole kilobytes");
  static_assert(RING <= 160 * 1024, "the rings fit a CU's LDS");
};
using Tile256 = TileShape<2, 4, 4, 2, 2, 4, 2, 3, true>;
using Tile256x192 = TileShape<4, 2, 2, 3, 2, 4, 2, 4, true>;
using Tile256x128 = TileShape<4, 2, 2, 2, 3, 4, 2, 4, true>;
using Tile128 = TileShape<2, 4, 2, 1, 4, 8, 2>;
// beside readers (read_weights), where what is copied comes from the L2s, four more waves that only copy: those that multiply
// then wait for no copy to be taken (2,048 x 1,600 x 6,400 51.1 -> 47.0 us, 150 x 4,800 x 1,600 13.6 -> 12.6; without readers 0 to 5 % slower)
using Tile128Fed = TileShape<2, 4, 2, 1, 4, 8, 3, 4, false, 4>;
using Tile128Pair = TileShape<2, 4, 2, 1, 2, 8, 4>;  // two blocks a CU (pairs_of_blocks below)
using Tile64x128 = TileShape<2, 4, 1, 1, 3, 8, 4>;  // two blocks a CU, as the next
using Tile32x128 = TileShape<1, 4, 1, 1, 4, 8, 2>;

// Weights read ahead by compute units that have no tile.  A compute unit gets some 25 to 40 GB/s of what its die's L2 does not hold, and
// the k-blocks of a column of tiles are such to each block that meets them first: with weights from memory 333 x 4,800 x 1,600 (tiles
// of 128 x 128, 114 blocks) took 16.5 us, out of the last-level cache 13.4, however many slots the ring had.  So blocks behind the
// tiles', as many a die as it has units left, read their die's columns in the order in which the tiles will want them, four pieces of a k-block on their way
// each, into nothing: the tiles' copies find them in the L2.  They end by themselves with the last piece and nobody waits for
// them.  us, rows x features x K, without and with: 333 x 6,400 x 1,600 16.7 -> 14.4, 2,048 x 1,600 x 6,400 53.7 -> 47.1, 1,000 x 1,600 x 1,600 (64 x 128)
// 13.3 -> 10.6, 200 x 4,800 x 1,600 (64 x 128) 13.8 -> 10.9, 100 x 5,440 x 1,024 (32 x 128) 8.1 -> 7.3.
template <typename S>
__device__ __forceinline__ void read_weights(const GemmArgs& p, int kb_lo, int n_blocks) {
  const int tiles_n = (p.N + S::BN - 1) / S::BN;
  const int reader = ((int)blockIdx.x - p.tile_blocks) / N_DIES, readers = ((int)gridDim.x - p.tile_blocks) / N_DIES;
  int first, columns;
  if (!columns_of_die<S::PANEL>((p.M + S::BM - 1) / S::BM, tiles_n, blockIdx.x % N_DIES, first, columns)) return;
  columns = min(columns, readers);  // (a reader that had more to read would still be at it when the tiles are done)
  const int n_fb = (p.N + 15) / 16, pieces = n_blocks * columns;  // a k-block of a column of tiles
  constexpr int LOADS = (S::BN * 8 + S::THREADS - 1) / S::THREADS, GROUP = 4;
  for (int i = reader; i < pieces; i += GROUP * readers) {
    u32x4_t v[GROUP][LOADS];
#pragma unroll
    for (int g = 0; g < GROUP; ++g) {
      const int at = min(i + g * readers, pieces - 1), kb = kb_lo + at / columns, fb = (first + at % columns) % tiles_n * (S::BN / 16);
#pragma unroll
      for (int l = 0; l < LOADS; ++l) {
        const int t = min(l * S::THREADS + (int)threadIdx.x, S::BN * 8 - 1);
        v[g][l] = *(const u32x4_t*)(p.W + ((size_t)min(fb + (t >> 7), n_fb - 1) * p.w_kblocks + kb) * 1024 + (t & 127) * 8);
      }
    }
#pragma unroll
    for (int g = 0; g < GROUP; ++g)
#pragma unroll
      for (int l = 0; l < LOADS; ++l) asm volatile("" ::"v"(v[g][l]));  // (read, and forgotten)
  }
}

// Pipeline: k-block kb is multiplied out of one slot of each ring while the next ones are on their way into
// the others (lds_copy.h); one wait by count and one barrier a k-block.  Nothing passes through registers but the operands,
// which are read a quarter of a k-block (16 columns) ahead of their products: left to the compiler, each read stood next
// to its product (2,048 x 4,800 x 1,600: 36.0 us, 34.0 read ahead; 8,000 x 1,600 x 6,400: 178.7 and 167.0).  Before, the k-blocks went through
// registers into LDS two ahead: 42.6 and 192 us for these, 65 against 58.6 for 2,048 x 1,600 x 6,400, and where few
// rows give few tiles, so that a tile's own walk is the time, 39.0 against 14.0 for 333 x 1,600 x 6,400 and 14.8 against
// 7.1 for 333 x 1,600 x 1,600 (K in three parts; rows x features x K, weights from memory, on an MI355X).
// SPLIT: K is shared out over blockIdx.y and the partial sums go to the workspace (a kernel of
// its own, so that the unsplit one carries none of it).
// PACKED: W lies in the decode kernels' packed order.
template <typename S, bool SPLIT, bool PACKED>
__global__ __launch_bounds__(S::THREADS, S::WAVES_PER_SIMD) void gemm_bf16_tile_kernel(GemmArgs p) {
  constexpr int BM = S::BM, BN = S::BN, TM = S::TM, TN = S::TN, PA = S::PA, PB = S::PB;
  // (one buffer: the epilogue uses it again for the output tiles)
  __shared__ __attribute__((aligned(1024))) uint16_t smem[S::RING / 2];

  if (PACKED && (int)blockIdx.x >= p.tile_blocks) {
    const int lo = SPLIT ? blockIdx.y * p.blocks_per_split : 0, all = (p.K + BK - 1) / BK;
    return read_weights<S>(p, lo, SPLIT ? min(all, lo + p.blocks_per_split) - lo : all);
  }
  int tm, tn;
  if (!tile_of_block<S::PANEL>((p.M + BM - 1) / BM, (p.N + BN - 1) / BN, tm, tn)) return;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / S::WAVES_N, wn = wave % S::WAVES_N;
  const int m0 = tm * BM;
  const int n0 = tn * BN;

  f32x16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  // this split's k-blocks (all of them without a split)
  const int kb_lo = SPLIT ? blockIdx.y * p.blocks_per_split : 0;
  const int n_blocks = SPLIT ? min((p.K + BK - 1) / BK, kb_lo + p.blocks_per_split) - kb_lo : (p.K + BK - 1) / BK;

  // What this wave copies: rows of 128 bytes, eight of them a copy.  Row r's piece s of 16 bytes in LDS is piece
  // s ^ (r / 2 % 8) of the row in memory, so that lanes which read one piece of sixteen neighbouring rows meet sixteen
  // different groups of banks (s ^ (r % 8), which gives only eight, made a read take twice as long).  Packed weights need none of that: half a tile of 16 features x 64 k is a copy as it lies, and
  // sixteen lanes read 256 bytes in a row.  Rows beyond the matrix lie beyond the buffer's end, columns beyond K are
  // sent there.
  const int asker = S::COPIERS ? wave - S::WAVES : wave;
  const i32x4_t a_buf = copy_buffer(p.A, ((size_t)(p.M - 1) * p.lda + p.K) * 2);
  const i32x4_t b_buf = copy_buffer(p.W, PACKED ? (size_t)((p.N + 15) / 16) * p.w_kblocks * 2048
                                                : ((size_t)(p.N - 1) * p.ldw + p.K) * 2);
  const int row8 = lane >> 3;
  auto piece_of = [&](int copy) __attribute__((always_inline)) { return (lane & 7) ^ ((copy & 1) * 4 + (row8 >> 1)); };
  uint32_t a_from[PA], b_from[PB];
#pragma unroll
  for (int i = 0; i < PA; ++i) {
    const int row = m0 + (asker * PA + i) * 8 + row8;
    a_from[i] = row < p.M ? (uint32_t)(((size_t)row * p.lda + piece_of(asker * PA + i) * 8) * 2) : COPY_NOTHING;
  }
#pragma unroll
  for (int i = 0; i < PB; ++i) {
    const int g = asker * PB + i;
    if constexpr (PACKED) {
      const int fb = n0 / 16 + (g >> 1);
      b_from[i] = fb < (p.N + 15) / 16 ? (uint32_t)(((size_t)fb * p.w_kblocks * 1024 + (g & 1) * 512 + lane * 8) * 2) : COPY_NOTHING;
    } else {
      const int row = n0 + g * 8 + row8;
      b_from[i] = row < p.N ? (uint32_t)(((size_t)row * p.ldw + piece_of(g) * 8) * 2) : COPY_NOTHING;
    }
  }
  const uint32_t ring = lds_address(smem);
  const uint32_t a_to = ring + asker * PA * 1024, b_to = ring + S::B_BASE + asker * PB * 1024;
  // What a round asks for: rows' k-block ka into slot sa and weights' k-block kb into slot sb, copy by copy.
  // (k-blocks beyond the last are asked for too, as nothing: the waits then count the same copies in every round)
  struct Round {
    int k_left_a, k_left_b;  // columns from the k-block on
    uint32_t a_at, a_k, b_at, b_k;
  };
  auto round_of = [&](int ka, int sa, int kb, int sb) __attribute__((always_inline)) {
    Round q;
    q.k_left_a = ka < n_blocks ? p.K - (kb_lo + ka) * BK : 0;
    q.k_left_b = S::ALIKE ? q.k_left_a : kb < n_blocks ? p.K - (kb_lo + kb) * BK : 0;
    q.a_at = (uint32_t)sa * S::A_STRIDE, q.b_at = S::ALIKE ? q.a_at : (uint32_t)sb * S::B_STRIDE;
    q.a_k = (uint32_t)(kb_lo + ka) * (BK * 2), q.b_k = (uint32_t)(kb_lo + kb) * (BK * 2 * (PACKED ? 16 : 1));
    return q;
  };
  auto ask = [&](const Round& q, int i) __attribute__((always_inline)) {
    if (i < PA) {
      copy16_to_lds(a_buf, piece_of(asker * PA + i) * 8 < q.k_left_a ? a_from[i < PA ? i : 0] : COPY_NOTHING, q.a_k, a_to + q.a_at + i * 1024);
    } else {
      const int j = i < PA ? 0 : i - PA;
      copy16_to_lds(b_buf, (PACKED ? q.k_left_b > 0 : piece_of(asker * PB + j) * 8 < q.k_left_b) ? b_from[j] : COPY_NOTHING, q.b_k,
                    b_to + q.b_at + j * 1024);
    }
  };

  const int row32 = lane & 31, hi = lane >> 5;
  const char* const a_row = (const char*)smem + (wm * TM * 32 + row32) * 128;
  const char* const b_row = (const char*)smem + S::B_BASE +
                            (PACKED ? ((wn * TN * 2 + (row32 >> 4)) * 2 + hi) * 1024 + (row32 & 15) * 16 : (wn * TN * 32 + row32) * 128);

  // Without a split the tiles are accumulated transposed (the weights' rows as the MFMA's rows):
  // a lane then holds four neighbouring columns of one output row, which the epilogue wants.
  auto mfma_tile = [](const bf16x8_t& a, const bf16x8_t& b, const f32x16_t& c) __attribute__((always_inline)) {
    if constexpr (SPLIT)
      return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_f32_32x32x16_bf16(b, a, c, 0, 0, 0);
  };
  // The operands of 16 columns (a quarter of a k-block) go to registers one quarter ahead of their products, also
  // across the barrier: a k-block's last quarter is multiplied after the barrier that lets the next one be read.
  bf16x8_t fa[2][TM], fb[2][TN];
  int slot_a = 0;
  [[maybe_unused]] int slot_b = 0;
  auto read_quarter = [&](int set, int q) __attribute__((always_inline)) {
    const char* af = a_row + slot_a * S::A_STRIDE;
    const char* bf = b_row + (S::ALIKE ? slot_a : slot_b) * S::B_STRIDE;
    const int s = ((2 * q + hi) ^ ((row32 >> 1) & 7)) * 16;
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[set][i] = *(const bf16x8_t*)(af + i * 32 * 128 + s);
#pragma unroll
    for (int j = 0; j < TN; ++j) fb[set][j] = *(const bf16x8_t*)(PACKED ? bf + j * 4096 + q * 256 : bf + j * 32 * 128 + s);
    __builtin_amdgcn_sched_barrier(0);
  };
  // The products of a quarter; with SPREAD copies `from` up to `to` of a round go between them.
  constexpr int TAKES = S::SPREAD ? (S::COPIES + 1) / 2 : S::COPIES;  // copies asked for beside a quarter's products, or at once
  auto multiply = [&](int set, const Round& round, int from, int to) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        acc[i][j] = mfma_tile(fa[set][i], fb[set][j], acc[i][j]);
        const int done = i * TN + j, n = to - from;
        if ((done + 1) * n / (TM * TN) > done * n / (TM * TN)) {
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int c = done * n / (TM * TN); c < (done + 1) * n / (TM * TN); ++c) ask(round, from + c);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    __builtin_amdgcn_sched_barrier(0);
  };

  constexpr int SA = S::SLOTS_A, SB = S::SLOTS_B, AHEAD = SA > SB ? SA : SB;
  if constexpr (S::COPIERS > 0) {
    static_assert(S::ALIKE && !S::SPREAD, "waves that only copy");
    if (wave >= S::WAVES) {
#pragma unroll
      for (int t = 0; t < SA - 1; ++t) {
        const Round q = round_of(t, t, t, t);
#pragma unroll
        for (int i = 0; i < S::COPIES; ++i) ask(q, i);
      }
      for (int kb = 0; kb < n_blocks; ++kb) {
        copies_arrived<(SA - 2) * S::COPIES>();
        ring_barrier();  // k-block kb is whole, and nobody reads the slot of k-block kb - 1 any more
        const int next = slot_a == 0 ? SA - 1 : slot_a - 1;
        const Round q = round_of(kb + SA - 1, next, kb + SA - 1, next);
#pragma unroll
        for (int i = 0; i < S::COPIES; ++i) ask(q, i);
        slot_a = slot_a == SA - 1 ? 0 : slot_a + 1;
      }
      copies_arrived<0>();  // (what was asked for beyond the end: the epilogue writes where it goes)
      if (!SPLIT) __syncthreads();
      return;
    }
    const Round none = round_of(0, 0, 0, 0);
    for (int kb = 0; kb < n_blocks; ++kb) {
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      ring_barrier();
      read_quarter(0, 0);
      if (kb > 0) multiply(1, none, 0, 0);
      read_quarter(1, 1);
      multiply(0, none, 0, 0);
      read_quarter(0, 2);
      multiply(1, none, 0, 0);
      read_quarter(1, 3);
      multiply(0, none, 0, 0);
      slot_a = slot_a == SA - 1 ? 0 : slot_a + 1;
    }
    multiply(1, none, 0, 0);
  } else {
#pragma unroll
    for (int t = 1 - AHEAD; t < 0; ++t) {  // as rounds before the first would have it
      const Round q = round_of(t + SA - 1, t + SA - 1, t + SB - 1, t + SB - 1);
#pragma unroll
      for (int i = t + SA - 1 >= 0 ? 0 : PA; i < (t + SB - 1 >= 0 ? S::COPIES : PA); ++i) ask(q, i);
    }
    // A round asks for rows SA - 1 and weights SB - 1 k-blocks ahead, the rows first.  When k-block kb begins, its rows came
    // with round kb - SA + 1 and its weights with round kb - SB + 1: so many copies were asked for behind both.
    constexpr int BEHIND_A = PB + (SA - 2) * S::COPIES, BEHIND_B = (SB - 2) * S::COPIES;
    const Round none = round_of(0, 0, 0, 0);
    for (int kb = 0; kb < n_blocks; ++kb) {
      copies_arrived<(BEHIND_A < BEHIND_B ? BEHIND_A : BEHIND_B)>();
      ring_barrier();  // k-block kb is whole, and nobody reads the slots of k-block kb - 1 any more
      read_quarter(0, 0);
      const int next_a = slot_a == 0 ? SA - 1 : slot_a - 1, next_b = S::ALIKE ? next_a : slot_b == 0 ? SB - 1 : slot_b - 1;
      const Round q = round_of(kb + SA - 1, next_a, kb + SB - 1, next_b);
      if (!S::SPREAD || kb == 0) {
#pragma unroll
        for (int i = 0; i < TAKES; ++i) ask(q, i);
        if (kb > 0) multiply(1, none, 0, 0);
      } else {
        multiply(1, q, 0, TAKES);
      }
      read_quarter(1, 1);
      multiply(0, q, TAKES, S::COPIES);
      read_quarter(0, 2);
      multiply(1, none, 0, 0);
      read_quarter(1, 3);
      multiply(0, none, 0, 0);
      slot_a = slot_a == SA - 1 ? 0 : slot_a + 1;
      if constexpr (!S::ALIKE) slot_b = slot_b == SB - 1 ? 0 : slot_b + 1;
    }
    multiply(1, none, 0, 0);
    copies_arrived<0>();  // (what was asked for beyond the end: the epilogue writes where it goes)
  }

  if constexpr (SPLIT) {  // the partial sums as they are; sum_partials adds them and runs the epilogue
    float* ws = p.ws + (size_t)blockIdx.y * p.M * p.N;
    const bool through = p.flags & FLAG_THROUGH;
    const __amdgpu_buffer_rsrc_t ws_buf = through_buffer(ws, (size_t)p.M * p.N * 4);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + wn * TN * 32 + j * 32 + (lane & 31);
      if (n >= p.N) continue;
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int mb = m0 + wm * TM * 32 + i * 32 + 4 * (lane >> 5);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int m = mb + 8 * (r >> 2) + (r & 3);
          if (m >= p.M) continue;
          if (through)
            store_through(ws_buf, (uint32_t)(((size_t)m * p.N + n) * 4), acc[i][j][r]);
          else
            ws[(size_t)m * p.N + n] = acc[i][j][r];
        }
      }
    }
    return;
  }

  // Epilogue.  Accumulator r of a transposed 32x32 tile: output row lane % 32, column
  // 8*(r/4) + 4*(lane/32) + r%4.  Stored like that, every lane of a store would be in
  // another row (and with the tiles not transposed, a store would be 64 bytes of 2-byte
  // pieces): the epilogue took 13 to 24 us of a product's 43 to 62 at 2,048 rows.  So each
  // wave passes its tile through LDS, 32 rows at a time, and takes it out again with eight
  // neighbouring columns a lane: stores of 16 or 32 bytes a lane that cover whole rows of
  // the wave's tile.  The region of a wave is its own; a wave's LDS accesses keep their order.
  constexpr int NW = S::WAVES;
  constexpr int WCOLS = TN * 32;   // columns of a wave's tile
  constexpr int EST = WCOLS + 4;   // floats a row in LDS: sixteen-byte pieces of neighbouring rows on other banks
  static_assert(NW * 32 * EST * 4 <= (int)sizeof(smem), "the waves' output tiles fit the k-blocks' LDS");
  __syncthreads();  // nobody reads a k-block any more
  float* const tile = (float*)smem + wave * 32 * EST;
  // (read and written through two names: an element is read and then written by the same lane,
  // and no load has to wait for stores to other elements)
  const float* __restrict__ res = (const float*)p.out;
  float* __restrict__ out_f = (float*)p.out;
  uint16_t* __restrict__ out_h = (uint16_t*)p.out;
  const bool f32_out = p.flags & (FLAG_ACCUMULATE | FLAG_OUT_F32);
  const bool through = p.flags & FLAG_THROUGH;
  const __amdgpu_buffer_rsrc_t out_buf = through_buffer(p.out, ((size_t)(p.M - 1) * p.ldo + p.N) * (f32_out ? 4 : 2));
  // CPL columns a lane on the way out, 16 bytes of the output: eight bfloat16 or four floats, so
  // that a store covers whole 128-byte lines of a few rows
  auto emit = [&](auto cpl) __attribute__((always_inline)) {
    constexpr int CPL = decltype(cpl)::value;
    constexpr int LPR = WCOLS / CPL;  // lanes a row
    constexpr int RPP = 64 / LPR;     // rows a pass
    constexpr int PASSES = (32 + RPP - 1) / RPP;
    constexpr int GROUP = PASSES < 32 / CPL ? PASSES : 32 / CPL;  // passes whose values are in registers at a time
    const int erow = lane / LPR, ecol = (lane % LPR) * CPL;
    const bool elane = erow < RPP;
    const int n = n0 + wn * WCOLS + ecol;  // this lane's columns, in every row it takes out
    float bias[CPL];
#pragma unroll
    for (int c = 0; c < CPL; ++c) bias[c] = p.bias ? p.bias[min(n + c, p.N - 1)] : 0.f;
    // whole pieces of 16 bytes: the row stride and the base keep them aligned, and all the columns exist
    const bool vec = n + CPL <= p.N && p.ldo % CPL == 0 && ((uintptr_t)p.out & 15) == 0;
    // this lane's columns are a key's or a value's: its pieces go to the token's place in the
    // cache pages (the host has seen to it that a piece of eight columns stays inside a head), through to memory
    // like the rest (left in the L2s until the kernel's end, the 13 MB of 2,048 rows of GPT-2 XL cost 1.3 us a layer:
    // 8,970 -> 8,909 us a step)
    const bool kv_lane = CPL == 8 && (p.flags & FLAG_KV) && n >= p.q_width;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int mt = m0 + wm * TM * 32 + i * 32;  // first row of this 32-row tile
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();  // every lane has read the tile before
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *(float4*)(tile + (lane & 31) * EST + j * 32 + 8 * g + 4 * (lane >> 5)) =
              make_float4(acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int s0 = 0; s0 < PASSES; s0 += GROUP) {
        // what is added to goes out first, all of the group's at once (left to itself the
        // compiler puts each load next to its use: one trip after another)
        float o[GROUP][CPL];
        if (p.flags & FLAG_ACCUMULATE) {
#pragma unroll
          for (int s = 0; s < GROUP; ++s) {
            const float* orow = res + (size_t)min(mt + (s0 + s) * RPP + erow, p.M - 1) * p.ldo;
            if (vec) {
              const float4 t = *(const float4*)(orow + n);  // (CPL is 4 with 32-bit outputs)
              o[s][0] = t.x, o[s][1] = t.y, o[s][2] = t.z, o[s][3] = t.w;
            } else {
#pragma unroll
              for (int c = 0; c < CPL; ++c) o[s][c] = orow[min(n + c, p.N - 1)];
            }
          }
        }
        uint16_t* place[GROUP];
        if (kv_lane) {
#pragma unroll
          for (int s = 0; s < GROUP; ++s) place[s] = kv_place(p, min(mt + (s0 + s) * RPP + erow, p.M - 1), n);
        }
        __builtin_amdgcn_sched_barrier(0);
        float v[GROUP][CPL];
#pragma unroll
        for (int s = 0; s < GROUP; ++s) {
          const int row = min((s0 + s) * RPP + erow, 31);
#pragma unroll
          for (int c = 0; c < CPL; c += 4) {
            const float4 t = *(const float4*)(tile + row * EST + ecol + c);
            v[s][c] = t.x + bias[c], v[s][c + 1] = t.y + bias[c + 1], v[s][c + 2] = t.z + bias[c + 2], v[s][c + 3] = t.w + bias[c + 3];
          }
        }
        if (p.flags & FLAG_ACCUMULATE) {
#pragma unroll
          for (int s = 0; s < GROUP; ++s)
#pragma unroll
            for (int c = 0; c < CPL; ++c) v[s][c] += o[s][c];
        } else if (p.flags & FLAG_GELU) {
#pragma unroll
          for (int s = 0; s < GROUP; ++s)
#pragma unroll
            for (int c = 0; c < CPL; ++c) v[s][c] = gelu_tanh_fast(v[s][c]);
        } else if (p.flags & FLAG_RELU2) {
#pragma unroll
          for (int s = 0; s < GROUP; ++s)
#pragma unroll
            for (int c = 0; c < CPL; ++c) v[s][c] = relu_squared(v[s][c]);
        }
#pragma unroll
        for (int s = 0; s < GROUP; ++s) {
          const int row = (s0 + s) * RPP + erow, m = mt + row;
          if (!elane || row >= 32 || m >= p.M || n >= p.N) continue;
          const size_t at = (size_t)m * p.ldo + n;
          if (vec) {
            u32x4_t t;
            if constexpr (CPL == 4)
              t = u32x4_t{__float_as_uint(v[s][0]), __float_as_uint(v[s][1]), __float_as_uint(v[s][2]), __float_as_uint(v[s][3])};
            else
              t = u32x4_t{pack_bf16x2(v[s][0], v[s][1]), pack_bf16x2(v[s][2], v[s][3]),
                          pack_bf16x2(v[s][4], v[s][5]), pack_bf16x2(v[s][6], v[s][7])};
            if (kv_lane)  // (the pieces of a head's row are neighbouring lanes': whole lines of the page)
              store_through(place[s], t);
            else if (through)
              store_through(out_buf, (uint32_t)(at * (CPL == 4 ? 4 : 2)), t);
            else
              *(u32x4_t*)(CPL == 4 ? (void*)(out_f + at) : (void*)(out_h + at)) = t;
          } else if (kv_lane) {
#pragma unroll
            for (int c = 0; c < CPL; ++c)
              if (n + c < p.N) place[s][c] = f32_to_bf16_bits(v[s][c]);
          } else {
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
              if (n + c >= p.N) break;
              if constexpr (CPL == 4)
                out_f[at + c] = v[s][c];
              else
                out_h[at + c] = f32_to_bf16_bits(v[s][c]);
            }
          }
        }
      }
    }
  };
  if (f32_out)
    emit(std::integral_constant<int, 4>{});
  else
    emit(std::integral_constant<int, 8>{});
}

// ---------------------------------------------------------------------------
// Skinny kernel: out^T tile = W[16 features, K] x A^T[K, up to 64 rows].
// Lane l of a wave reads 32 contiguous bytes of W row (l % 16) per 64-wide
// k-block, at k offset (l / 16) * 16, and feeds them to two 16x16x32 MFMAs;
// the activation fragment uses the same k offsets, so the products pair up.

#define SK_WAVES 4
#define SK_MAXM 64
// From 17 rows on the tile kernel takes the product, with K split over blocks where the tiles alone
// do not fill the GPU.  (A kernel that streamed the weights once for 17 to 64 rows, 64 features a
// block, was 3 to 17 % slower at GPT-2 XL's projections and twice as slow at the vocabulary's head.)
#define TILE_MIN_ROWS 17

template <int MT>  // number of 16-row groups of activations (1..4)
__global__ __launch_bounds__(256) void gemm_bf16_skinny_kernel(GemmArgs p) {
  __shared__ float red[SK_WAVES][MT][64 * 4];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int n0 = blockIdx.x * 16;
  const int wrow = n0 + (lane & 15);
  const int koff = (lane >> 4) * 16;
  const bool wvalid = wrow < p.N;
  const uint16_t* wrow_p = p.W + (size_t)(wvalid ? wrow : 0) * p.ldw;
  // packed weights: the lane's two pieces of a k-block are pieces 2 g and 2 g + 1 of its feature
  const uint16_t* wpack0 = p.W + packed_piece(wvalid ? wrow : 0, 2 * (lane >> 4), p.w_kblocks);
  const uint16_t* wpack1 = p.W + packed_piece(wvalid ? wrow : 0, 2 * (lane >> 4) + 1, p.w_kblocks);

  f32x4_t acc[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) acc[t] = (f32x4_t){0.f, 0.f, 0.f, 0.f};

  union Frag {
    uint4 u;
    bf16x8_t v;
  };

  for (int k0 = wave * 64; k0 < p.K; k0 += SK_WAVES * 64) {
    const int k = k0 + koff;  // this lane covers k .. k+15
    Frag w0, w1;
    const uint4 t0 = *(const uint4*)(p.w_packed ? wpack0 + (size_t)k0 * 16 : wrow_p + min(k, p.K - 8));
    const uint4 t1 = *(const uint4*)(p.w_packed ? wpack1 + (size_t)k0 * 16 : wrow_p + min(k + 8, p.K - 8));
    w0.u = (wvalid && k < p.K) ? t0 : ZERO4;
    w1.u = (wvalid && k + 8 < p.K) ? t1 : ZERO4;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      const int m = t * 16 + (lane & 15);
      const bool av = m < p.M;
      const uint16_t* arow = p.A + (size_t)(av ? m : 0) * p.lda;
      Frag a0, a1;
      const uint4 u0 = *(const uint4*)(arow + min(k, p.K - 8));
      const uint4 u1 = *(const uint4*)(arow + min(k + 8, p.K - 8));
      a0.u = (av && k < p.K) ? u0 : ZERO4;
      a1.u = (av && k + 8 < p.K) ? u1 : ZERO4;
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0.v, a0.v, acc[t], 0, 0, 0);
      acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1.v, a1.v, acc[t], 0, 0, 0);
    }
  }

  // sum the waves' partial tiles in a fixed order
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave][t][lane * 4 + r] = acc[t][r];
  __syncthreads();
  if (wave == 0) {
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      // accumulator r: feature row 4*(lane/16) + r, activation column lane%16
      const int m = t * 16 + (lane & 15);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < SK_WAVES; ++w) v += red[w][t][lane * 4 + r];
        const int n = n0 + 4 * (lane >> 4) + r;
        if (m < p.M && n < p.N) store_out(p, m, n, v);
      }
    }
  }
}

// ---------------------------------------------------------------------------

DEFINE_LAST_ERROR(mlxlm_last_error)

static int check_args(const GemmArgs& p) {
  if (p.M < 0 || p.N <= 0 || p.K <= 0) FAIL("gemm_bf16: bad sizes M=%d N=%d K=%d", p.M, p.N, p.K);
  if (p.K % 8 != 0) FAIL("gemm_bf16: K=%d must be a multiple of 8", p.K);
  if (p.lda % 8 != 0 || p.ldw % 8 != 0)
    FAIL("gemm_bf16: row strides lda=%d ldw=%d must be multiples of 8", p.lda, p.ldw);
  if (p.lda < p.K || (!p.w_packed && p.ldw < p.K) || p.ldo < p.N)
    FAIL("gemm_bf16: row strides smaller than the rows (lda=%d ldw=%d ldo=%d)", p.lda, p.ldw, p.ldo);
  if (!p.A || !p.W || !p.out) FAIL("gemm_bf16: null pointer");
  if (((uintptr_t)p.A | (uintptr_t)p.W) & 15) FAIL("gemm_bf16: A and W must be 16-byte aligned");
  const size_t w_elements = p.w_packed ? (size_t)((p.N + 15) / 16) * p.w_kblocks * 1024 : (size_t)p.N * p.ldw;
  if ((size_t)p.M * p.lda >= (1u << 31) || w_elements >= (1u << 31))
    FAIL("gemm_bf16: operands of 2^31 elements or more are not supported");
  if ((p.flags & FLAG_ACCUMULATE) && (p.flags & FLAG_ACT_ANY))
    FAIL("gemm_bf16: an activation and accumulate cannot be combined");
  if ((p.flags & FLAG_ACT_ANY) == FLAG_ACT_ANY) FAIL("gemm_bf16: two activations at once");
  return 0;
}

template <typename S, bool CAN_SPLIT>
static void launch_tiles(GemmArgs p, hipStream_t stream, int readers = 0) {
  const long tiles = (long)((p.M + S::BM - 1) / S::BM) * ((p.N + S::BN - 1) / S::BN);
  dim3 grid((unsigned)((tiles + 7) / 8 * 8), p.n_splits), block(S::THREADS);  // a run of tiles for each die
  p.tile_blocks = grid.x, grid.x += N_DIES * readers;
  if constexpr (CAN_SPLIT) {
    if (p.n_splits > 1) {
      if (p.w_packed)
        hipLaunchKernelGGL((gemm_bf16_tile_kernel<S, true, true>), grid, block, 0, stream, p);
      else
        hipLaunchKernelGGL((gemm_bf16_tile_kernel<S, true, false>), grid, block, 0, stream, p);
      return;
    }
  }
  if (p.w_packed)
    hipLaunchKernelGGL((gemm_bf16_tile_kernel<S, false, true>), grid, block, 0, stream, p);
  else
    hipLaunchKernelGGL((gemm_bf16_tile_kernel<S, false, false>), grid, block, 0, stream, p);
}

#define FEW_ROWS 64  // up to so many rows packed weights are other kernels' (gemm_bf16_decode.hip), but for a K that they do not hold

// Compute units of a die that a product's tiles leave idle, for each part of K, and the columns of tiles that they would read ahead for.
template <typename S>
static void idle_units(int M, int N, int n_splits, int* idle, double* columns) {
  const int tiles_m = (M + S::BM - 1) / S::BM, run = (tiles_m * ((N + S::BN - 1) / S::BN) + N_DIES - 1) / N_DIES;
  const int left = n_compute_units() / N_DIES - run * n_splits;
  *idle = left > 0 ? left / n_splits : 0;
  *columns = (double)run / (tiles_m < S::PANEL ? tiles_m : S::PANEL);
}

// Compute units a die and part of K that read the weights ahead (0: none do).  Too few of them fall behind the tiles and are still
// reading when those are done: 240 x 6,784 x 1,600 in tiles of 64 x 128 (five a die for seven columns) 14.2 -> 14.8 us, 536 x 1,600 x 1,600 in
// two parts (one for two) 8.8 -> 9.6; 240 x 6,400 x 1,600 (seven for six) 14.2 -> 12.0.  Tiles of 32 x 128 gain a little from any.  Tiles of 128 x 128 want one a column, of
// at most eight (480 x 6,400 x 1,600, seven for six, 17.0 -> 14.9, 352 x 7,680 x 1,600, nine for eight, 17.3 -> 15.0; 224 x 8,704 x 1,600, fifteen for nine of which eight are read,
// 17.3 -> 18.4, 96 x 10,880 x 1,600 17.8 -> 18.7), but where the last row of tiles is nearly empty they have less to gain and to spare (390 x 6,400 x
// 1,600 15.0 -> 15.4, 520 x 4,800 x 1,600, eight for five, 15.0 -> 15.2), so the line lies at nearly two a column: with one, prompts of 510 and 640 tokens of GPT-2 XL would take
// 1.4 and 0.6 % less (4,284 -> 4,230, 4,860 -> 4,833 us), of 390, 520 and 536 1.1, 0.9 and 0.6 % more, of large 520 2 % more and 640 1.2 % less; with one and
// a half 520 and 536 0.7 % more and 640 0.5 % less.  2,048 x 1,600 x 1,600 (1.85 a column) 16.5 -> 15.5, x 6,400 53.5 -> 48.2.  They
// gain nothing in parts of K (25 us with 24.6 for 536 x 1,600 x 6,400 in two); the widest were
// level or behind (1,000 x 6,400 x 1,600 in 256 x 128 24.7 -> 25.7).  More than eight (twelve) take from the tiles: 333 x 6,400 x 1,600 15.2 with twelve, 14.1 with eight.
static int readers_of(int variant, int M, int N, int n_splits, bool packed) {
  int idle = 0;
  double columns = 0.0;
  if (!packed || M <= FEW_ROWS || (variant == 1 && n_splits > 1)) return 0;
  if (variant == 1)
    idle_units<Tile128>(M, N, n_splits, &idle, &columns);
  else if (variant == 5)
    idle_units<Tile64x128>(M, N, n_splits, &idle, &columns);
  else if (variant == 6)
    idle_units<Tile32x128>(M, N, n_splits, &idle, &columns);
  else
    return 0;
  if (variant == 1 && columns > 8.0) return 0;
  const double enough = variant == 1 ? 1.83 : 0.9;
  const int most = variant == 1 ? 8 : 12;
  return idle < 1 || idle < enough * columns ? 0 : idle < most ? idle : most;
}

// Whether they keep up with the tiles, so that those cost what fed ones do.  Tiles of 64 rows: where there is a reader for each column (65 x 10,880 x 2,048, ten
// for eleven, 0.42 us a k-block; 160 x 8,192 x 2,048, eight for eight, 0.35).  Of 32 rows, which take half as long: from five readers for four columns on
// (65 x 8,192 x 6,144, eight for eight, 0.31; 100 x 6,144 x 2,048, eight for six, 0.25; 65 x 6,400 x 1,600, thirteen for six, 0.23); with three or fewer, as parts
// of K leave them, from nine for four on (65 x 1,600 x 6,400 in four parts, three for five thirds, 0.31; 100 x 1,280 x 5,120 in four, three for five quarters, 0.21) or
// two for one (80 x 768 x 3,072 in six, 0.22).
static bool readers_keep_up(int variant, int M, int N, int n_splits) {
  if (!readers_of(variant, M, N, n_splits, true)) return false;
  int idle = 0;
  double columns = 0.0;
  if (variant == 5) {
    idle_units<Tile64x128>(M, N, n_splits, &idle, &columns);
    return idle >= columns;
  }
  if (variant == 6) {
    idle_units<Tile32x128>(M, N, n_splits, &idle, &columns);
    return idle >= (idle > 3 ? 1.25 : columns > 1.0 ? 2.25 : 2.0) * columns;
  }
  return true;
}

// What a shape costs, in microseconds: `launch` once, `tile` for each round of tiles on a CU and `kblock` for each k-block of it, `pair`
// a k-block where two blocks share the CU (shapes that fit twice); where CUs that have no tile read weights ahead and keep up, `fed_tile` and
// `fed` instead.  `full`: what a k-block costs at least where all CUs ask the L2s for one at once (fewer in proportion); `full_alone` with K whole and nobody who
// reads ahead (128 x 128, K whole: 500 x 8,192 x 6,144 0.60, 2,048 x 2,048 x 5,440 0.55; 900 x 1,280 x 5,120 in three parts, which are stored as they are, 0.77).
// Fitted to the times of 18 numbers of rows from 65 to 2,048 against 18 matrices of widths 768 to 2,048, K up to
// 6,400, weights from 2.5 GB of memory, each with K in 1 to 8 parts; the shape and parts chosen from these prices are within 0.6 % of the best on average (at
// worst 1.13 times; the prices before the readers, 6.7 % and 1.76).  Fifteen numbers of rows against fourteen matrices up to 16,384 x 8,192: 1.1 %, at worst 1.2 times.
struct TilePrice {
  int variant, bm, bn, per_cu;
  double launch, tile, kblock, pair;
  bool splits;  // K may be split over blocks
  double fed_tile, fed, full, full_alone;
};
static const TilePrice TILE_PRICES[] = {
    {3, Tile256::BM, Tile256::BN, 1, 0.0, 7.69, 1.042, 0.0, false, 0.0, 0.0, 0.0, 0.0},
    {4, Tile256x192::BM, Tile256x192::BN, 1, 0.0, 6.9, 0.885, 0.0, false, 0.0, 0.0, 0.0, 0.0},
    {8, Tile256x128::BM, Tile256x128::BN, 1, 0.0, 6.1, 0.65, 0.0, false, 0.0, 0.0, 0.0, 0.0},
    {1, Tile128::BM, Tile128::BN, 1, 0.21, 4.09, 0.499, 0.0, true, 4.25, 0.331, 0.686, 0.6},
    {5, Tile64x128::BM, Tile64x128::BN, 2, 3.11, 1.32, 0.363, 0.708, true, 0.49, 0.32, 0.403, 0.403},
    {6, Tile32x128::BM, Tile32x128::BN, 2, 2.83, 1.54, 0.27, 0.516, true, 0.83, 0.202, 0.316, 0.316},
};
// Products that nobody reads ahead for: row-major weights, and up to 64 rows (what the kernels for few rows leave, a longer K than they hold).
// Fitted to 16 numbers of rows from 20 to 8,000.  us, rows x features x K, row-major, by these and by the prices above: 333 x 4,800 x 1,600 14.3 and 16.7,
// 150 x 6,400 x 1,600 12.5 and 14.6, 333 x 5,376 x 1,024 10.5 and 11.9, 65 x 10,880 x 2,048 18.0 and 19.7.
static const TilePrice UNFED_PRICES[] = {
    {3, Tile256::BM, Tile256::BN, 1, 0.0, 7.78, 1.3, 0.0, false, 0.0, 0.0, 0.0, 0.0},
    {4, Tile256x192::BM, Tile256x192::BN, 1, 0.0, 7.26, 1.0, 0.0, false, 0.0, 0.0, 0.0, 0.0},
    {8, Tile256x128::BM, Tile256x128::BN, 1, 0.0, 7.6, 0.7, 0.0, false, 0.0, 0.0, 0.0, 0.0},
    {1, Tile128::BM, Tile128::BN, 1, 0.0, 4.33, 0.49, 0.0, true, 0.0, 0.0, 0.0, 0.0},
    {5, Tile64x128::BM, Tile64x128::BN, 2, 0.52, 2.81, 0.38, 0.77, true, 0.0, 0.0, 0.0, 0.0},
    {6, Tile32x128::BM, Tile32x128::BN, 2, 1.81, 1.98, 0.33, 0.52, true, 0.0, 0.0, 0.0, 0.0},
};

static double price(const TilePrice& s, int M, int N, int K, int n_splits, bool packed) {
  const long tiles = (long)((M + s.bm - 1) / s.bm) * ((N + s.bn - 1) / s.bn), cus = n_compute_units(), per_die = cus / N_DIES;
  const long n = ((tiles + N_DIES - 1) / N_DIES * n_splits + per_die - 1) / per_die;  // the busiest CU
  const int k_blocks = ((K + BK - 1) / BK + n_splits - 1) / n_splits;
  const bool fed = packed && readers_keep_up(s.variant, M, N, n_splits);
  const double least = (n_splits == 1 && !fed ? s.full_alone : s.full) * (tiles * n_splits < cus ? tiles * n_splits : cus) / cus;
  if (fed) return s.launch + s.fed_tile + k_blocks * (s.fed > least ? s.fed : least);
  if (n == 1) return s.launch + s.tile + k_blocks * (s.kblock > least ? s.kblock : least);
  if (s.per_cu == 1) return s.launch + n * (s.tile + k_blocks * s.kblock);
  return s.launch + (n / 2) * (s.tile + k_blocks * s.pair) + (n % 2) * (s.tile + k_blocks * s.kblock);
}
// The cheapest shape for K in so many parts, and its price.
static int cheapest_shape(int M, int N, int K, int n_splits, bool packed, double* us) {
  int variant = 0;
  const auto look = [&](const TilePrice& s) {
    if (n_splits > 1 && !s.splits) return;
    const double t = price(s, M, N, K, n_splits, packed);
    if (!variant || t < *us) variant = s.variant, *us = t;
  };
  if (M <= FEW_ROWS || !packed)
    for (const TilePrice& s : UNFED_PRICES) look(s);
  else
    for (const TilePrice& s : TILE_PRICES) look(s);
  return variant;
}

// Matrices of more columns of tiles than CUs (a vocabulary's) at rows that would leave half or more of the last 256-row
// tile empty: blocks of 128 x 128, two a CU, one of which reads weights or stores while the other multiplies.  The prices
// were fitted to narrower matrices and do not show it.  32-bit logits, us, by the prices and so: 50,257 x 768 at 65 / 128 /
// 333 rows 27.5 / 36.1 / 76.8 and 24.5 / 31.8 / 70.8 (26.3 / 33.7 / 66.1 with the kernel before the LDS ring, which had two
// such blocks a CU too); 50,257 x 1,600 43.0 / 53.6 / 107 and 38.9 / 49.3 / 106 (46.4 / 54.1 / 98.4); 50,304 x 1,024 26.5 / 31.5 /
// 60.7 and 24.3 / 27.6 / 55.1 (28.8 / 31.6 / 58.3).  Not at 170, 256 and 512 rows (50,257 x 768 40.4 / 47.3 / 86.3 and 46.8 / 56.3 /
// 98.4), nor where every CU has one tile (32,000 x 2,048 at 128 rows 30.8 and 36.9).
static bool pairs_of_blocks(int M, int N) {
  return ((M > 64 && M <= 128) || (M > 256 && M <= 384)) && (N + 127) / 128 > n_compute_units();
}

// Into how many parts the kernels with tiles 128 wide should split K (1: no split).  Few rows
// give few tiles (up to 128 rows of GPT-2 XL's projections are 13 to 50 tiles for 256 CUs), and a
// tile's walk through K takes the same time whether 50 or 500 of them run; a split shortens the
// walk and costs a second kernel that reads the partial sums ([parts][M][N] floats).  Both sides
// are priced: the walk as above, the second kernel as a launch plus its bytes at 3 TB/s.
// `fused`: the second kernel stands in for one that would run anyway (the norm that follows a
// sum into the residual stream, the write of keys and values into their pages), so it costs only
// the extra bytes.  A part keeps three k-blocks or more, and more parts have to be 2 % cheaper.  Where the second kernel would run anyway, more parts
// of twelve k-blocks or more that all have a unit to themselves may cost 5 % more by these prices: in steps they are level or ahead (GPT-2 XL, us a step, 72 rows of
// 1,600 x 6,400 in 5 / 6 / 8 parts 2,632 / 2,630 / 2,630, 200 rows in two and four 3,200 and 3,156; large, 260 rows of 1,280 x 5,120 in two and three 2,316 and
// 2,206), at worst 0.7 % behind (150 rows of 1,600 x 6,400 in four and six 2,887 and 2,908).
// `force` > 0 asks for that many parts wherever K has them (for tests of small sizes).  `ws_floats`: what the parts' sums
// have to fit.  (Priced for packed weights; row-major ones, which only direct callers have, go in as many parts, so that both orders give the same bits.)
extern "C" int gemm_bf16_parts(int M, int N, int K, int fused, int force, size_t ws_floats) {
  if (M < TILE_MIN_ROWS) return 1;
  const int n_blocks = (K + BK - 1) / BK;
  int best = 1;
  if (force > 0) {
    best = force < n_blocks ? force : n_blocks;
  } else {
    constexpr int MOST = 16;
    const size_t fit = ws_floats / ((size_t)M * N);
    const int most = fit < MOST ? (int)fit : MOST;
    double price_of[MOST + 1], best_us = 0.0;
    int last = 1;
    for (int s = 1; s == 1 || (s <= most && s <= n_blocks / 3); ++s) {
      double us = 0.0;
      cheapest_shape(M, N, K, s, true, &us);
      if (s > 1) us += (fused ? 1.0 : 2.5) + 8.0 * (fused ? s - 1 : s) * (double)M * N / 3e6;
      if (s == 1 || us < 0.98 * best_us) best = s, best_us = us;
      price_of[s] = us, last = s;
    }
    const long tiles = (long)((M + Tile64x128::BM - 1) / Tile64x128::BM) * ((N + Tile64x128::BN - 1) / Tile64x128::BN);
    if (fused && best > 1)
      for (int s = best + 1; s <= last && tiles * s <= n_compute_units() && n_blocks >= 12 * s; ++s)
        if (price_of[s] < 1.05 * best_us) best = s;
  }
  if (best <= 1) return 1;
  const int per = (n_blocks + best - 1) / best;
  return (n_blocks + per - 1) / per;  // no empty part
}

extern "C" int gemm_bf16_splits(int M, int N, int K, int fused, int force) { return gemm_bf16_parts(M, N, K, fused, force, SIZE_MAX); }

// The kernel (`variant` below) for a product with K whole.
extern "C" int gemm_bf16_shape(int M, int N, int K, int packed) {
  double us = 0.0;
  return M < TILE_MIN_ROWS ? 2 : pairs_of_blocks(M, N) ? 7 : cheapest_shape(M, N, K, 1, packed, &us);
}

// variant: 0 = choose, 1 = 128 x 128 tiles, 7 = the same two blocks a CU, 2 = skinny kernel, 3 = 256 x 256 tiles, 4 = 256 x 192
// tiles, 5 = 64 x 128 tiles, 6 = 32 x 128 tiles, 8 = 256 x 128 tiles.  n_splits > 1 (variants 1, 5 and 6 only): no
// epilogue, the partial sums go to ws.  ldw == 0: W is in the decode kernels' packed order
// (tiles of 16 features x 64 k, zero padded), which all kernels here read as well as rows.
extern "C" int gemm_bf16_scatter(void* out, const void* A, const void* W, const float* bias, int M, int N,
                                 int K, int lda, int ldw, int ldo, int flags, int variant, int n_splits,
                                 float* ws, size_t ws_floats, void* k_pages, void* v_pages, size_t page_stride,
                                 const int* block_table, int max_blocks, const int* token_req,
                                 const int* positions, int q_width, int kv_width, int head_dim, int page_size,
                                 hipStream_t stream);

extern "C" int gemm_bf16(void* out, const void* A, const void* W, const float* bias, int M, int N,
                         int K, int lda, int ldw, int ldo, int flags, int variant, int n_splits,
                         float* ws, size_t ws_floats, hipStream_t stream) {
  return gemm_bf16_scatter(out, A, W, bias, M, N, K, lda, ldw, ldo, flags, variant, n_splits, ws, ws_floats,
                           nullptr, nullptr, 0, nullptr, 0, nullptr, nullptr, 0, 0, 0, 0, stream);
}

// The same with the cache scatter of a fused q/k/v projection (k_pages != null, no split of K, a
// bfloat16 output): the columns from q_width on (kv_width of keys, then kv_width of values) of
// row m go to position positions[m] of request token_req[m] in the pages, through the block
// table, and are not written to out.
extern "C" int gemm_bf16_scatter(void* out, const void* A, const void* W, const float* bias, int M, int N,
                                 int K, int lda, int ldw, int ldo, int flags, int variant, int n_splits,
                                 float* ws, size_t ws_floats, void* k_pages, void* v_pages, size_t page_stride,
                                 const int* block_table, int max_blocks, const int* token_req,
                                 const int* positions, int q_width, int kv_width, int head_dim, int page_size,
                                 hipStream_t stream) {
  GemmArgs p;
  p.A = (const uint16_t*)A;
  p.W = (const uint16_t*)W;
  p.bias = bias;
  p.out = out;
  p.M = M, p.N = N, p.K = K;
  p.lda = lda, p.ldw = ldw, p.ldo = ldo;
  p.flags = flags & (FLAG_ACT_ANY | FLAG_ACCUMULATE | FLAG_OUT_F32);
  p.w_packed = ldw == 0 ? 1 : 0, p.w_kblocks = (K + BK - 1) / BK;
  if (check_args(p)) return 1;
  if (M == 0) return 0;
  p.k_pages = (uint16_t*)k_pages, p.v_pages = (uint16_t*)v_pages, p.page_stride = page_stride;
  p.block_table = block_table, p.token_req = token_req, p.positions = positions;
  p.max_blocks = max_blocks, p.q_width = q_width, p.kv_width = kv_width, p.head_dim = head_dim, p.page_size = page_size;
  if (k_pages) {
    if (flags & (FLAG_ACT_ANY | FLAG_ACCUMULATE | FLAG_OUT_F32)) FAIL("gemm_bf16: the cache scatter goes with a plain bfloat16 output");
    if (n_splits > 1) FAIL("gemm_bf16: with K split, sum_partials scatters keys and values");
    if (!v_pages || !block_table || !token_req || !positions)
      FAIL("gemm_bf16: the cache scatter needs pages, block table, token_req and positions");
    if (head_dim <= 0 || page_size <= 0 || head_dim % 8 != 0 || q_width % 8 != 0 || kv_width % head_dim != 0 ||
        q_width + 2 * kv_width != N)
      FAIL("gemm_bf16: q_width %d + 2 * kv_width %d must be N=%d, widths multiples of 8, kv_width of head_dim %d",
           q_width, kv_width, N, head_dim);
    if (page_stride % 8 != 0 || (((uintptr_t)k_pages | (uintptr_t)v_pages) & 15))
      FAIL("gemm_bf16: cache pages must be 16-byte aligned");
    if (ldo < q_width) FAIL("gemm_bf16: ldo=%d smaller than q_width=%d", ldo, q_width);
    p.flags |= FLAG_KV;
  }
  const int n_blocks = (K + BK - 1) / BK;
  if (n_splits < 1 || n_splits > n_blocks) FAIL("gemm_bf16: %d splits of K=%d", n_splits, K);
  p.ws = ws, p.n_splits = n_splits, p.blocks_per_split = (n_blocks + n_splits - 1) / n_splits;
  if (fits_through_buffer((size_t)M * ldo * 4) && fits_through_buffer((size_t)M * N * 4)) p.flags |= FLAG_THROUGH;
  if (n_splits > 1) {
    double us = 0.0;
    if (variant == 0) variant = cheapest_shape(M, N, K, n_splits, p.w_packed, &us);
    if (variant != 1 && variant != 5 && variant != 6) FAIL("gemm_bf16: only the tiles of 128, 64 and 32 rows by 128 split K");
    if (p.blocks_per_split * (n_splits - 1) >= n_blocks) FAIL("gemm_bf16: %d splits of K=%d leave one empty", n_splits, K);
    if (!ws || ((uintptr_t)ws & 15) || ws_floats < (size_t)n_splits * M * N)
      FAIL("gemm_bf16: %d splits of %d x %d need an aligned workspace of that many floats", n_splits, M, N);
  }
  if (variant == 0) variant = gemm_bf16_shape(M, N, K, p.w_packed);
  if (variant == 2) {
    if (M > SK_MAXM) FAIL("gemm_bf16: the skinny kernel takes at most %d rows, got %d", SK_MAXM, M);
    dim3 grid((N + 15) / 16), block(256);
    const int mt = (M + 15) / 16;
    if (mt == 1)
      hipLaunchKernelGGL(gemm_bf16_skinny_kernel<1>, grid, block, 0, stream, p);
    else if (mt == 2)
      hipLaunchKernelGGL(gemm_bf16_skinny_kernel<2>, grid, block, 0, stream, p);
    else if (mt == 3)
      hipLaunchKernelGGL(gemm_bf16_skinny_kernel<3>, grid, block, 0, stream, p);
    else
      hipLaunchKernelGGL(gemm_bf16_skinny_kernel<4>, grid, block, 0, stream, p);
  } else if (variant == 1) {
    const int readers = readers_of(variant, M, N, n_splits, p.w_packed);
    if (readers && n_splits == 1)
      launch_tiles<Tile128Fed, false>(p, stream, readers);
    else
      launch_tiles<Tile128, true>(p, stream, readers);
  } else if (variant == 7) {
    launch_tiles<Tile128Pair, false>(p, stream);
  } else if (variant == 5) {
    launch_tiles<Tile64x128, true>(p, stream, readers_of(variant, M, N, n_splits, p.w_packed));
  } else if (variant == 6) {
    launch_tiles<Tile32x128, true>(p, stream, readers_of(variant, M, N, n_splits, p.w_packed));
  } else if (variant == 3) {
    launch_tiles<Tile256, false>(p, stream);
  } else if (variant == 4) {
    launch_tiles<Tile256x192, false>(p, stream);
  } else if (variant == 8) {
    launch_tiles<Tile256x128, false>(p, stream);
  } else {
    FAIL("gemm_bf16: unknown variant %d", variant);
  }
  CHECK_LAUNCH("gemm_bf16");
  return 0;
}
