// Linear layer on float operands with float sums:
//   out[m, n] = epilogue( sum_k A[m, k] * W[n, k] + bias[n] )
// A is [M, K], W is [N, K], both contiguous along k.  Epilogues: plain,
// tanh-GELU, or accumulate into the residual stream.  Any M, N; K % 4 == 0.
// The 32-bit twin of gemm_bf16.hip; replaces the same nn.Linear calls
// (mlx_lm/models/gpt2.py:41-42,52,68,76-80,167).
//
// Three ways, chosen by rows and prices: up to 64 rows a kernel that streams the weights once and tiles of few blocks both multiply with
// v_mfma_f32_16x16x4_f32, a sixteenth of bfloat16's rate; where tiles are many, each float is cut into two half-precision
// numbers (23 or 24 of its 24 bits) and three products of them stand for one, with smaller errors against 64 bits than the former; sums
// for which a row's range is too wide for that are computed with the float instruction.
//
// Up to 64 rows (decode steps) take a kernel of their own, which streams W
// once through v_mfma_f32_16x16x4_f32, 16 features a block: a 64 x 64 tile
// would spend its time on rows that are not there and leave most compute units
// without a block.  Where 16 features a block still give fewer blocks than
// units, K goes in parts and a second kernel (the caller's) adds them up.
#include "common.h"
#include "lds_copy.h"
#include "tile_order.h"

#define FLAG_GELU FLAG_ACT_GELU
#define FLAG_RELU2 FLAG_ACT_RELU2  // the square of the ReLU instead
#define FLAG_ACCUMULATE 2

// What a row is scaled by where it is cut, a power of two, and the sum (as scaled) below which its small values are in doubt (cut_rows_kernel).
struct RowScale {
  int up;
  float doubt;
};

struct GemmArgs {
  const float* A;
  const float* W;
  const float* bias;
  float* out;
  int M, N, K;
  int lda, ldw, ldo;
  int flags;
  // blockIdx.y takes part y of K's chunks of 64 columns (`per_split` of them) and leaves its sums
  // in ws[y][ws_rows][N], without bias or epilogue
  int n_splits, per_split, ws_rows;
  float* ws;
  // the tiles' rows, cut (cut_rows_kernel), ldc floats apart, and the rows' and features' scales
  const float* cut;
  const RowScale* a_scales;
  const RowScale* w_scales;
  int ldc;
  int through;  // out and a part of ws are below 4 GB: the tiles' stores go through to memory
  // the kernel for few rows: the features from q_width on are keys and values, which go to their pages too (k_pages null:
  // none do)
  float* k_pages;
  float* v_pages;
  size_t page_stride;
  const int* block_table;
  const int* token_req;
  const int* positions;
  int max_blocks, q_width, kv_width, head_dim, page_size;
};

// Where feature n (from q_width on) of row m lies in its page.
__device__ __forceinline__ float* page_place(const GemmArgs& p, int m, int n) {
  const int c = n - p.q_width, cc = c < p.kv_width ? c : c - p.kv_width, head = cc / p.head_dim;
  const int pos = p.positions[m], page = p.block_table[(size_t)p.token_req[m] * p.max_blocks + pos / p.page_size];
  return (c < p.kv_width ? p.k_pages : p.v_pages) + (size_t)page * p.page_stride + ((size_t)head * p.page_size + pos % p.page_size) * p.head_dim +
         (cc - head * p.head_dim);
}

// Many rows: WAVES_M x WAVES_N waves a block, each with TM x TN tiles of 16 x 16 outputs.
// v_mfma_f32_16x16x4_f32 computes D = A B for A 16 x 4 and B 4 x 16: lane l brings A[l % 16][l / 16] and
// B[l / 16][l % 16] and gets D[4 * (l / 16) + r][l % 16] in accumulator r.  Here A is the weights' tile and B the
// rows', so that a lane holds four neighbouring features of one row.  Which column of k an instruction's four slots
// stand for is free as long as both operands agree, so a lane reads 16 bytes, columns 4 * (l / 16) .. + 3 of each 16,
// and the four floats go to four instructions.
//
// Steps of 32 columns (rows of 128 bytes) are copied straight into a ring of slots in LDS, two ahead (lds_copy.h); a
// row's 16-byte pieces lie permuted as in gemm_bf16.hip, so that sixteen neighbouring rows meet sixteen groups of banks.
// At 32-bit speed (a sixteenth of bfloat16's) a step of 64 x 128 outputs is 2,048 cycles of each SIMD's matrix unit and
// 24 KB of copies: the matrix units are the bound, and what is lost is lost to CUs that hold fewer tiles than others.
// Hence small tiles, two blocks a CU, and K in parts where that evens the blocks out (`price`).  (The kernel before
// this one read its operands from the L2s in the instruction's layout, sixteen pieces of 64 bytes a load, and had no
// parts: 1,050 rows against GPT-2 large's four matrices took 178, 76, 179 and 287 us, now 87, 36, 117 and 113, the last
// with K in three; the library's rate for a large product would make them 68, 22, 90 and 90.)
template <int WAVES_M_, int WAVES_N_, int TM_, int TN_>
struct F32Shape {
  static constexpr int WAVES_M = WAVES_M_, WAVES_N = WAVES_N_, TM = TM_, TN = TN_;
  static constexpr int WAVES = WAVES_M * WAVES_N, THREADS = 64 * WAVES, STAGES = 3, STEP = 32;
  static constexpr int BM = WAVES_M * TM * 16, BN = WAVES_N * TN * 16;
  static constexpr int PA = BM / 8 / WAVES, PB = BN / 8 / WAVES, COPIES = PA + PB;  // copies of eight rows a wave and step
  static constexpr int STAGE_BYTES = (BM + BN) * STEP * 4;
  static_assert(BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0, "a wave copies whole kilobytes");
};
using F32Tile64x128 = F32Shape<2, 2, 2, 4>;
using F32Tile64 = F32Shape<2, 2, 2, 2>;
using F32Tile32x64 = F32Shape<2, 2, 1, 2>;

template <typename S>
__global__ __launch_bounds__(S::THREADS, 2) void gemm_f32_tile_kernel(GemmArgs p) {
  constexpr int BM = S::BM, BN = S::BN, TM = S::TM, TN = S::TN, PA = S::PA, PB = S::PB, STAGES = S::STAGES;
  __shared__ __attribute__((aligned(1024))) float smem[STAGES * S::STAGE_BYTES / 4];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int x = lane & 15, g = lane >> 4;
  const int wm = wave / S::WAVES_N, wn = wave % S::WAVES_N;
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int k_lo = blockIdx.z * p.per_split * 64, k_end = min(p.K, k_lo + p.per_split * 64);
  const int n_steps = (k_end - k_lo + S::STEP - 1) / S::STEP;

  // the block's rows and features, each a buffer of its own from the block's first on: what lies beyond the matrix lies
  // beyond the buffer, or is sent there
  const int a_rows = min(BM, p.M - m0), b_rows = min(BN, p.N - n0);
  const i32x4_t a_buf = copy_buffer(p.A + (size_t)m0 * p.lda, ((size_t)(a_rows - 1) * p.lda + p.K) * 4);
  const i32x4_t b_buf = copy_buffer(p.W + (size_t)n0 * p.ldw, ((size_t)(b_rows - 1) * p.ldw + p.K) * 4);
  const int row8 = lane >> 3;
  auto piece_of = [&](int copy) __attribute__((always_inline)) { return (lane & 7) ^ ((copy & 1) * 4 + (row8 >> 1)); };
  uint32_t a_from[PA], b_from[PB];
#pragma unroll
  for (int i = 0; i < PA; ++i) {
    const int c = wave * PA + i, row = c * 8 + row8;
    a_from[i] = row < a_rows ? (uint32_t)(((size_t)row * p.lda + piece_of(c) * 4) * 4) : COPY_NOTHING;
  }
#pragma unroll
  for (int i = 0; i < PB; ++i) {
    const int c = wave * PB + i, row = c * 8 + row8;
    b_from[i] = row < b_rows ? (uint32_t)(((size_t)row * p.ldw + piece_of(c) * 4) * 4) : COPY_NOTHING;
  }
  const uint32_t ring = lds_address(smem);
  // (steps beyond the last are asked for too, as nothing: the waits then count the same copies in every round)
  auto ask = [&](int t, int slot) __attribute__((always_inline)) {
    const int k = k_lo + t * S::STEP, left = t < n_steps ? k_end - k : 0;
    const uint32_t k4 = t < n_steps ? (uint32_t)k * 4u : 0u, at = ring + (uint32_t)slot * S::STAGE_BYTES;
#pragma unroll
    for (int i = 0; i < PA; ++i)
      copy16_to_lds(a_buf, piece_of(wave * PA + i) * 4 < left ? a_from[i] : COPY_NOTHING, k4, at + (wave * PA + i) * 1024);
#pragma unroll
    for (int i = 0; i < PB; ++i)
      copy16_to_lds(b_buf, piece_of(wave * PB + i) * 4 < left ? b_from[i] : COPY_NOTHING, k4, at + BM * 128 + (wave * PB + i) * 1024);
  };

  f32x4_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const char* const a_row = (const char*)smem + (wm * TM * 16 + x) * 128;
  const char* const b_row = (const char*)smem + BM * 128 + (wn * TN * 16 + x) * 128;
  // the operands of 16 columns go to registers that many columns ahead of their products, also across the barrier
  f32x4_t fa[2][TM], fb[2][TN];
  auto read_half = [&](int h, int slot) __attribute__((always_inline)) {
    const int s = ((4 * h + g) ^ (x >> 1)) * 16;
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[h][i] = *(const f32x4_t*)(a_row + slot * S::STAGE_BYTES + i * 2048 + s);
#pragma unroll
    for (int j = 0; j < TN; ++j) fb[h][j] = *(const f32x4_t*)(b_row + slot * S::STAGE_BYTES + j * 2048 + s);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto multiply = [&](int h) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[h][j][c], fa[h][i][c], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t) ask(t, t);
  int slot = 0;
  for (int t = 0; t < n_steps; ++t) {
    copies_arrived<(STAGES - 2) * S::COPIES>();
    ring_barrier();  // step t is whole, and nobody reads the slot of step t - 1 any more
    read_half(0, slot);
    ask(t + STAGES - 1, slot == 0 ? STAGES - 1 : slot - 1);
    if (t > 0) multiply(1);
    read_half(1, slot);
    multiply(0);
    slot = slot == STAGES - 1 ? 0 : slot + 1;
  }
  multiply(1);
  copies_arrived<0>();  // (what was asked for beyond the end)

  // Epilogue.  Accumulator r of tile (i, j): row 16 * i + x, feature 16 * j + 4 * g + r.  What is read (bias, the
  // residual stream to add to) is read for a row of tiles before anything of it is stored: a load that comes after a
  // store to memory it might alias waits for it.
  const bool parts = p.n_splits > 1;
  float* const out = parts ? p.ws + (size_t)blockIdx.z * p.ws_rows * p.N : p.out;
  const int ldo = parts ? p.N : p.ldo;
  const bool vec = ldo % 4 == 0 && ((uintptr_t)out & 15) == 0;
  // (through to memory, as far as a buffer reaches: 1,050 x 1,280 x 5,120 in three parts 114.8 -> 113.5 us, two parts of
  // 1,280 columns 34.7 -> 33.9, the wide ones level)
  const __amdgpu_buffer_rsrc_t out_buf = through_buffer(out, ((size_t)(p.M - 1) * ldo + p.N) * 4);
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + (wm * TM + i) * 16 + x;
    if (m >= p.M) continue;
    f32x4_t v[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + (wn * TN + j) * 16 + 4 * g;
      v[j] = acc[i][j];
      if (parts) continue;
      const bool add = p.flags & FLAG_ACCUMULATE, whole = vec && n + 4 <= p.N;
      f32x4_t old = {0.f, 0.f, 0.f, 0.f};
      if (add && whole) old = *(const f32x4_t*)(p.out + (size_t)m * ldo + n);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int nc = min(n + r, p.N - 1);
        const float b = p.bias ? p.bias[nc] : 0.f;
        if (add)
          v[j][r] = (whole ? old[r] : p.out[(size_t)m * ldo + nc]) + (v[j][r] + b);
        else
          v[j][r] = activate<false>(p.flags, v[j][r] + b);
      }
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + (wn * TN + j) * 16 + 4 * g;
      if (vec && n + 4 <= p.N) {
        if (p.through)
          store_through(out_buf, (uint32_t)(((size_t)m * ldo + n) * 4), __builtin_bit_cast(u32x4_t, v[j]));
        else
          *(f32x4_t*)(out + (size_t)m * ldo + n) = v[j];
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (n + r < p.N) out[(size_t)m * ldo + n + r] = v[j][r];
      }
    }
  }
}

// Many rows, cut operands.  x = 2^-s (h + 2^-12 l), h the half-precision number nearest to 2^s x and l the one nearest to 2^12 times what h
// leaves: 11 bits each and a sign, so that the two are x's 24 bits in three of four cases and miss by its last one in the fourth.  x y is then
// h h' + 2^-12 (h l' + l h'), three of v_mfma_f32_32x32x16_f16 (16 times the rate of the float instruction: 5 times its products); 2^-24 l l', 2^-22 of x y at
// most, is left out.  One power of two a row of A and of W puts the row's greatest value between 2^14 and 2^15: values down to 2^-28 below it
// then keep both halves whole (LEAST_WHOLE).  Of smaller ones a row counts how many there are, and a sum that is not well above what they can have lost
// (one great value beside them that met a zero, say) is computed again with the 32-bit instructions (the end of gemm_f32_cut_kernel).
// h h' and the two smaller products are summed apart, each 16 columns an instruction, so a sum is rounded a
// quarter as often as with the float instruction (4 columns each): 2-norm of the error over the result's, normal rows against weights of 0.02,
// K = 768 / 1,280 / 5,120, 1.9e-7 / 2.4e-7 / 4.6e-7 against 5.0e-7 / 6.4e-7 / 1.3e-6 (the same of rows that a GELU left, and 2.2e-7 / 2.8e-7 / 5.4e-7 against 5.7e-7 /
// 7.4e-7 / 1.5e-6 with one column a thousand times the others); largest error over the sum of magnitudes, in 2^-24, 1.5 to 2.7 against
// 4.3 to 9.3 (K from 256 to 6,400, 65 to 4,000 rows).  At K = 16 the cut's own error shows (8.6e-8 against 7.4e-8), hence CUT_FROM_K.
//
// cut_rows_kernel finds the powers and lays the rows out cut, a row's octet of columns as 16 bytes of h and 16 of l where its 32
// bytes were, so that a tile copies both operands alike; the features' are found beside them, by each call: what is kept is
// wrong as soon as a caller changes its weights in place.  (The product finds the weights in the last-level cache then: from 600 rows on it takes no time, at 120
// to 200 rows 1 to 4 % of a step, which the prices' last term leaves to other tiles where those are as good.)  The weights, which would
// take as much memory again, are cut in registers, 16 columns ahead of their products (28 vector instructions for 8 columns of 32 features, between
// a wave's products); six products of three bfloat16 numbers each, exact without scales, took 106 us instead of 68 for 1,050 x 5,120 x 1,280.
//
// What bounds it: at 2,048 rows and more the power (with zeros instead of numbers 4,096 x 4,096 x 1,280 takes three quarters of the time), below
// the tiles' number and what a CU gets out of the L2s.  us, rows x features x K, with the launch that cuts (weights from memory) and in brackets with the float
// instruction's tiles: 300 x 3,840 x 1,280 31.8 (37.2), 1,050 x 3,840 x 1,280 54 (93), 1,050 x 5,120 x 1,280 73 (114), 1,050 x 1,280 x 5,120 in five parts 71.5 (111),
// 2,048 x 6,400 x 1,600 167 (316: 133 -> 251 TFLOP/s).  Where blocks are few the launch ahead is not made up for: 200 x 1,280 x 1,280 15.5 (13.3), 1,050 x 768 x 768
// 20.2 (18.8); `price` draws the line.  Where every sum is computed again, 1,050 x 5,120 x 1,280 takes 390.
//
// Four waves a block, WAVES_M of them one below the other, each with TM x TN tiles of 32 x 32 outputs.  Side by side, so that each feature is cut by one
// wave only: with two by two, each cutting twice as many, 1,050 x 5,120 x 1,280 76.5, x 3,840 x 1,280 59.7, 300 x 3,840 x 1,280 36.5 us.
template <int WAVES_M_, int TM_, int TN_, int STAGES_, int PANEL_>
struct CutShape {
  static constexpr int WAVES_M = WAVES_M_, WAVES_N = 4 / WAVES_M_;
  static constexpr int TM = TM_, TN = TN_, STAGES = STAGES_, PANEL = PANEL_, WAVES = 4, THREADS = 256, STEP = 32;
  static constexpr int BM = WAVES_M * TM * 32, BN = WAVES_N * TN * 32;
  static constexpr int PA = BM / 8 / WAVES, PB = BN / 8 / WAVES, COPIES = PA + PB;  // copies of eight rows a wave and step
  static constexpr int STAGE_BYTES = (BM + BN) * STEP * 4;
};
using CutTile128 = CutShape<1, 4, 1, 2, 8>;
using CutTile64x128 = CutShape<1, 2, 1, 3, 8>;
using CutTile64 = CutShape<2, 1, 1, 3, 8>;

// Columns from which operands may be cut.
#define CUT_FROM_K 256
// The low halves are held so much greater: 2^15 at most beside a high half of 2^15.
#define LOW_UP 4096.f

typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

// Two floats as two half-precision numbers each: the one nearest to the scaled float and LOW_UP times what it leaves.
__device__ __forceinline__ void cut_pair(float x0, float x1, float scale, float low_scale, uint32_t& high, uint32_t& low) {
  const f16x2_t h = __builtin_convertvector((hw_f32x2_t{x0 * scale, x1 * scale}), f16x2_t);
  const f16x2_t l = {(_Float16)__builtin_fmaf((float)h.x, -LOW_UP, x0 * low_scale), (_Float16)__builtin_fmaf((float)h.y, -LOW_UP, x1 * low_scale)};
  high = __builtin_bit_cast(uint32_t, h), low = __builtin_bit_cast(uint32_t, l);
}
struct Cut {
  u32x4_t high, low;  // eight halves each
};
__device__ __forceinline__ Cut cut(f32x4_t a, f32x4_t b, float scale) {
  const float low_scale = scale * LOW_UP;
  uint32_t h[4], l[4];
  cut_pair(a.x, a.y, scale, low_scale, h[0], l[0]), cut_pair(a.z, a.w, scale, low_scale, h[1], l[1]);
  cut_pair(b.x, b.y, scale, low_scale, h[2], l[2]), cut_pair(b.z, b.w, scale, low_scale, h[3], l[3]);
  return Cut{u32x4_t{h[0], h[1], h[2], h[3]}, u32x4_t{l[0], l[1], l[2], l[3]}};
}
__device__ __forceinline__ f32x16_t mfma(u32x4_t a, u32x4_t b, f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}
// The tanh form of GELU (gelu_tanh of common.h) in sixteen instructions: x / (1 + 2^t), t = x (c1 + c2 x^2) with the product's rounding put right
// behind the hardware's exponential, the quotient by the hardware's reciprocal and what it leaves.  (Written with expf and a division it is some forty-five:
// 1,050 x 5,120 x 1,280 with bias 77.4 us and 75.0 so, 2,048 x 6,400 x 1,600 172.7 and 168.2; without an activation 71.8 and 167.)  Error against 64 bits, greatest and mean of the result, against gelu_tanh's: -3 to 3 4.4e-7 and 5.3e-8 (8.9e-7
// and 6.8e-8), -12 to 12 6.4e-6 and 2.7e-7 (1.0e-5 and 3.4e-7), 1e-6 to 1 1.2e-7 and 2.8e-8 (1.3e-7 and 2.8e-8); infinities, NaN and sums beyond every
// exponential give what they give there (infinity, NaN for minus infinity, -0).
__device__ __forceinline__ float gelu_tanh_short(float x) {
  constexpr double c = -2.0 * 0.79788456080286535588 * 1.44269504088896340736;  // -2 sqrt(2 / pi) log2 e
  constexpr float c1 = (float)c, c2 = (float)(c * 0.044715);
  const float p = __builtin_fmaf(x * x, c2, c1), t = x * p, rest = __builtin_fmaf(x, p, -t);
  const float e = __builtin_amdgcn_exp2f(t), right = __builtin_fmaf(e, rest * 0.6931471805599453f, e);
  const float d = 1.0f + (right == right ? right : e);  // (NaN: infinite t or e)
  const float r = __builtin_amdgcn_rcpf(d), q = x * r, left = __builtin_fmaf(-d, q, x);
  return fabsf(left) > 0.f ? __builtin_fmaf(left, r, q) : q;  // (nothing left, or NaN: infinite d or x)
}
__device__ __forceinline__ bool finite(float v) { return (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u; }
__device__ __forceinline__ float power_of_2(int e) { return __uint_as_float((uint32_t)(e + 127) << 23); }

// From here on up a scaled value's two halves hold it to 2^-23 of itself.  Below, half precision's least step leaves out 2^-37, and the low
// parts' product 2^-36 of what it is multiplied with (2^15 at most): 1.5 2^-21 a value.  A sum of 4 for each such value of its row and feature is
// then good to 1.5 2^-23 of itself; one below that is in doubt.
#define LEAST_WHOLE 0x1p-14f
#define DOUBT_A_VALUE 4.f

// Ahead of the products: the rows' greatest values, whose exponents say what a row is scaled by (so that its greatest
// value lies from 2^14 up to 2^15), how many of their values are small, and A's rows scaled and cut.  A's first, a block a row, which stays in registers up to 8,192 columns.  A cut row has
// the place of the row itself: where eight floats were lie eight high halves and eight low ones, up to whole steps of 32 columns.  (A wave a row, read
// twice: 1,050 x 5,120 12.5 us; 10.2 so, 2,048 x 6,400 in 6 us less, 1,280 columns 5.4 either way.)  Then the features, a wave each, read once but for those that have
// small values: they come from memory, which is what bounds this.  (Features a block each: with the product 200 x 4,800 x 1,600 36.2 us, 35.0 so, 1,050 x 1,280 x 1,280
// in two parts 29.7 and 29.0, prompts of 400 and 1,000 tokens of GPT-2 large 6,130 and 5,965, 10,270 and 10,150.)
struct CutArgs {
  const float* A;
  const float* W;
  int M, N, K, lda, ldw, ldc;
  u32x4_t* cut;
  RowScale* scales;  // [M], then [N]
};
// How a row is scaled whose greatest value has these bits (without the sign).
__device__ __forceinline__ int scale_up(uint32_t most) {
  const int e = (int)(most >> 23);
  return most == 0 || e == 255 ? 0 : min(14 + 127 - e, 115);  // (LOW_UP times the power is a float too)
}
// A wave a feature.
__device__ __forceinline__ void scale_of_feature(const CutArgs& p, int n, int lane) {
  if (n >= p.N) return;
  const float* from = p.W + (size_t)n * p.ldw;
  constexpr int HELD = 8;
  auto each = [&](auto see) __attribute__((always_inline)) {
    for (int k0 = 4 * lane; k0 < p.K; k0 += 256 * HELD) {
      f32x4_t v[HELD];
#pragma unroll
      for (int i = 0; i < HELD; ++i) {
        v[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (k0 + 256 * i < p.K) v[i] = *(const f32x4_t*)(from + k0 + 256 * i);
      }
#pragma unroll
      for (int i = 0; i < HELD; ++i)
#pragma unroll
        for (int c = 0; c < 4; ++c) see(v[i][c]);
    }
  };
  uint32_t most = 0, least = ~0u;  // (the least value that is not zero, less one)
  each([&](float v) __attribute__((always_inline)) {
    const uint32_t bits = __float_as_uint(v) & 0x7fffffffu;
    most = max(most, bits), least = min(least, bits - 1u);
  });
#pragma unroll
  for (int d = 32; d; d >>= 1) most = max(most, (uint32_t)__shfl_xor((int)most, d, 64)), least = min(least, (uint32_t)__shfl_xor((int)least, d, 64));
  const int up = scale_up(most);
  const float scale = power_of_2(up);
  int small = 0;
  if (least != ~0u && __uint_as_float(least + 1u) * scale < LEAST_WHOLE)  // (hardly ever)
    each([&](float v) __attribute__((always_inline)) { small += v != 0.f && fabsf(v * scale) < LEAST_WHOLE; });
#pragma unroll
  for (int d = 32; d; d >>= 1) small += __shfl_xor(small, d, 64);
  if (lane == 0) p.scales[p.M + n] = RowScale{up, most == 0 ? -INFINITY : DOUBT_A_VALUE * (float)small};
}
__global__ __launch_bounds__(256) void cut_rows_kernel(CutArgs p) {
  __shared__ uint32_t wave_most[4];
  __shared__ int n_small;
  const int row = blockIdx.x, tid = threadIdx.x;
  if (row >= p.M) return scale_of_feature(p, (row - p.M) * 4 + (tid >> 6), tid & 63);
  const float* from = p.A + (size_t)row * p.lda;
  constexpr int HELD = 4, CHUNK = 256 * 8 * HELD;
  f32x4_t v[HELD][2];
  auto load = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < HELD; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int k = k0 + (tid + 256 * i) * 8 + 4 * h;
        v[i][h] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if (k < p.K) v[i][h] = *(const f32x4_t*)(from + k);
      }
  };
  // (without their signs floats are ordered as integers are, infinities and NaN behind all others)
  uint32_t most = 0;
  for (int k0 = 0; k0 < p.K; k0 += CHUNK) {
    load(k0);
#pragma unroll
    for (int i = 0; i < HELD; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int c = 0; c < 4; ++c) most = max(most, __float_as_uint(v[i][h][c]) & 0x7fffffffu);
  }
#pragma unroll
  for (int d = 32; d; d >>= 1) most = max(most, (uint32_t)__shfl_xor((int)most, d, 64));
  if ((tid & 63) == 0) wave_most[tid >> 6] = most;
  if (tid == 0) n_small = 0;
  __syncthreads();
  most = max(max(wave_most[0], wave_most[1]), max(wave_most[2], wave_most[3]));
  const int up = scale_up(most);
  const float scale = power_of_2(up);
  u32x4_t* to = p.cut + (size_t)row * (p.ldc / 4);
  int small = 0;
  for (int k0 = 0; k0 < p.ldc; k0 += CHUNK) {
    if (p.K > CHUNK) load(k0);
#pragma unroll
    for (int i = 0; i < HELD; ++i) {
      const int k = k0 + (tid + 256 * i) * 8;
      if (k0 + 2048 * i >= p.ldc) break;
      if (k >= p.ldc) continue;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int c = 0; c < 4; ++c) small += v[i][h][c] != 0.f && fabsf(v[i][h][c] * scale) < LEAST_WHOLE;
      const Cut c = cut(v[i][0], v[i][1], scale);
      to[k / 4] = c.high, to[k / 4 + 1] = c.low;
    }
  }
  if (small) atomicAdd(&n_small, small);
  __syncthreads();
  if (tid == 0) p.scales[row] = RowScale{up, most == 0 ? -INFINITY : DOUBT_A_VALUE * (float)n_small};
}

template <typename S>
__global__ __launch_bounds__(S::THREADS, 2) void gemm_f32_cut_kernel(GemmArgs p) {
  constexpr int BM = S::BM, BN = S::BN, TM = S::TM, TN = S::TN, PA = S::PA, PB = S::PB, STAGES = S::STAGES;
  __shared__ __attribute__((aligned(1024))) float smem[STAGES * S::STAGE_BYTES / 4];
  __shared__ __attribute__((aligned(16))) RowScale scales[BM + BN];  // the tile's rows', then its features'
  int tm, tn;
  if (!tile_of_block<S::PANEL>((p.M + BM - 1) / BM, (p.N + BN - 1) / BN, tm, tn)) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int x = lane & 31, hi = lane >> 5;
  const int wm = wave / S::WAVES_N, wn = wave % S::WAVES_N;
  const int m0 = tm * BM, n0 = tn * BN;
  const int k_lo = blockIdx.y * p.per_split * 64, k_end = min(p.K, k_lo + p.per_split * 64);
  const int n_steps = (k_end - k_lo + S::STEP - 1) / S::STEP;

  // the block's rows and features, each a buffer of its own from the block's first on: what lies beyond the matrix lies
  // beyond the buffer, or is sent there
  const int a_rows = min(BM, p.M - m0), b_rows = min(BN, p.N - n0);
  const i32x4_t a_buf = copy_buffer(p.cut + (size_t)m0 * p.ldc, (size_t)a_rows * p.ldc * 4);
  const i32x4_t b_buf = copy_buffer(p.W + (size_t)n0 * p.ldw, ((size_t)(b_rows - 1) * p.ldw + p.K) * 4);
  const int row8 = lane >> 3;
  auto piece_of = [&](int copy) __attribute__((always_inline)) { return (lane & 7) ^ ((copy & 1) * 4 + (row8 >> 1)); };
  uint32_t a_from[PA], b_from[PB];
#pragma unroll
  for (int i = 0; i < PA; ++i) {
    const int c = wave * PA + i, row = c * 8 + row8;
    a_from[i] = row < a_rows ? (uint32_t)(((size_t)row * p.ldc + piece_of(c) * 4) * 4) : COPY_NOTHING;
  }
#pragma unroll
  for (int i = 0; i < PB; ++i) {
    const int c = wave * PB + i, row = c * 8 + row8;
    b_from[i] = row < b_rows ? (uint32_t)(((size_t)row * p.ldw + piece_of(c) * 4) * 4) : COPY_NOTHING;
  }
  const uint32_t ring = lds_address(smem);
  // (steps beyond the last are asked for too, as nothing: the waits then count the same copies in every round)
  auto ask = [&](int t, int slot) __attribute__((always_inline)) {
    const int k = k_lo + t * S::STEP, left = t < n_steps ? k_end - k : 0;
    const uint32_t k4 = t < n_steps ? (uint32_t)k * 4u : 0u, at = ring + (uint32_t)slot * S::STAGE_BYTES;
#pragma unroll
    for (int i = 0; i < PA; ++i)
      copy16_to_lds(a_buf, left > 0 ? a_from[i] : COPY_NOTHING, k4, at + (wave * PA + i) * 1024);
#pragma unroll
    for (int i = 0; i < PB; ++i)
      copy16_to_lds(b_buf, piece_of(wave * PB + i) * 4 < left ? b_from[i] : COPY_NOTHING, k4, at + BM * 128 + (wave * PB + i) * 1024);
  };

  static_assert(BM + BN <= S::THREADS, "a scale a thread");
  // (read behind the first step's wait and barrier)
  if ((int)threadIdx.x < BM + BN) {
    const int n = n0 + (int)threadIdx.x - BM;
    RowScale s = {0, -INFINITY};
    if ((int)threadIdx.x < a_rows) s = p.a_scales[m0 + threadIdx.x];
    if ((int)threadIdx.x >= BM && n < p.N) s = p.w_scales[n];
    scales[threadIdx.x] = s;
  }
  float scale[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) scale[j] = power_of_2(p.w_scales[min(n0 + (wn * TN + j) * 32 + x, p.N - 1)].up);

  // the products of the high parts, and those with a low part
  f32x16_t acc[TM][TN], low[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = low[i][j][r] = 0.f;
  const char* const a_row = (const char*)smem + (wm * TM * 32 + x) * 128;
  const char* const b_row = (const char*)smem + BM * 128 + (wn * TN * 32 + x) * 128;
  // the operands of 16 columns go to registers that many columns ahead of their products, also across the barrier
  Cut a[2][TM], b[2][TN];
  f32x4_t raw[TN][2];
  auto read_half = [&](int h, int slot) __attribute__((always_inline)) {
    const int s0 = ((4 * h + 2 * hi) ^ ((x >> 1) & 7)) * 16, s1 = s0 ^ 16;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      raw[j][0] = *(const f32x4_t*)(b_row + slot * S::STAGE_BYTES + j * 4096 + s0);
      raw[j][1] = *(const f32x4_t*)(b_row + slot * S::STAGE_BYTES + j * 4096 + s1);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      a[h][i].high = *(const u32x4_t*)(a_row + slot * S::STAGE_BYTES + i * 4096 + s0);
      a[h][i].low = *(const u32x4_t*)(a_row + slot * S::STAGE_BYTES + i * 4096 + s1);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  auto cut_half = [&](int h) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < TN; ++j) b[h][j] = cut(raw[j][0], raw[j][1], scale[j]);
  };
  auto multiply = [&](int h) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = mfma(b[h][j].high, a[h][i].high, acc[i][j]);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) low[i][j] = mfma(b[h][j].high, a[h][i].low, low[i][j]);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) low[i][j] = mfma(b[h][j].low, a[h][i].high, low[i][j]);
  };
#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t) ask(t, t);
  int slot = 0;
  for (int t = 0; t < n_steps; ++t) {
    copies_arrived<(STAGES - 2) * S::COPIES>();
    ring_barrier();  // step t is whole, and nobody reads the slot of step t - 1 any more
    read_half(0, slot);
    ask(t + STAGES - 1, slot == 0 ? STAGES - 1 : slot - 1);
    if (t > 0) multiply(1);
    cut_half(0);
    __builtin_amdgcn_sched_barrier(0);
    read_half(1, slot);
    multiply(0);
    cut_half(1);
    __builtin_amdgcn_sched_barrier(0);
    slot = slot == STAGES - 1 ? 0 : slot + 1;
  }
  multiply(1);
  copies_arrived<0>();  // (what was asked for beyond the end)

  // A row's sums leave their scales behind.  What is not finite or in doubt is computed again with the 32-bit instructions, out of the
  // operands themselves: an infinity's parts would give NaN, and the sums' own infinities and NaN come out as those instructions have them.
  // (Two sums of every other column, so that each is rounded as seldom as with the instruction of four columns.)
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    RowScale w_scale[16];
    float w_doubt = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      w_scale[r] = scales[BM + (wn * TN + j) * 32 + 8 * (r >> 2) + 4 * hi + (r & 3)];
      w_doubt = fmaxf(w_doubt, w_scale[r].doubt);
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const RowScale a_scale = scales[(wm * TM + i) * 32 + x];
      float least = INFINITY, nothing = 0.f;
      f32x16_t s;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s[r] = __builtin_fmaf(low[i][j][r], 1.f / LOW_UP, acc[i][j][r]);
        least = fminf(least, fabsf(s[r]));
        nothing = __builtin_fmaf(s[r], 0.f, nothing);
        acc[i][j][r] = ldexpf(s[r], -a_scale.up - w_scale[r].up);
      }
      if (__any(!(nothing == 0.f && least >= a_scale.doubt + w_doubt))) {
        f32x16_t sum[2];
#pragma unroll
        for (int r = 0; r < 16; ++r) sum[0][r] = sum[1][r] = 0.f;
        const float* ap = p.A + (size_t)min(m0 + (wm * TM + i) * 32 + x, p.M - 1) * p.lda;
        const float* wp = p.W + (size_t)min(n0 + (wn * TN + j) * 32 + x, p.N - 1) * p.ldw;
        for (int k0 = k_lo; k0 < k_end; k0 += 32) {
          f32x4_t av[4], wv[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const int k = k0 + 8 * q + 4 * hi;
            av[q] = wv[q] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            if (k < k_end) av[q] = *(const f32x4_t*)(ap + k), wv[q] = *(const f32x4_t*)(wp + k);
          }
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int c = 0; c < 4; ++c) sum[c & 1] = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[q][c], av[q][c], sum[c & 1], 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (!finite(s[r]) || fabsf(s[r]) < a_scale.doubt + w_scale[r].doubt) acc[i][j][r] = sum[0][r] + sum[1][r];
      }
    }
  }

  // Epilogue.  Accumulator r of tile (i, j): row 32 * i + x, feature 32 * j + 8 * (r / 4) + 4 * hi + r % 4.  What is read (bias, the
  // residual stream to add to) is read for a tile before anything of it is stored: a load that comes after a
  // store to memory it might alias waits for it.
  const bool parts = p.n_splits > 1;
  float* const out = parts ? p.ws + (size_t)blockIdx.y * p.ws_rows * p.N : p.out;
  const int ldo = parts ? p.N : p.ldo;
  const bool vec = ldo % 4 == 0 && ((uintptr_t)out & 15) == 0;
  const bool add = p.flags & FLAG_ACCUMULATE;
  // (Stores that leave their lines in the caches: through to memory, as the other tiles' are, a prompt of 1,000 tokens of GPT-2 large in float32 took
  // 11,170 us instead of 10,770, of XL 20,850 instead of 19,970; 1,050 x 5,120 x 1,280 alone 75.2 and 71.9.)
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int nt = n0 + (wn * TN + j) * 32 + 4 * hi;
    f32x4_t bias[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      bias[g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if (!p.bias || parts) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) bias[g][r] = p.bias[min(nt + 8 * g + r, p.N - 1)];
    }
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = m0 + (wm * TM + i) * 32 + x;
      if (m >= p.M) continue;
      f32x4_t v[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int n = nt + 8 * g;
        v[g] = f32x4_t{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
        if (parts) continue;
        const bool whole = vec && n + 4 <= p.N;
        f32x4_t old = {0.f, 0.f, 0.f, 0.f};
        if (add && whole) old = *(const f32x4_t*)(p.out + (size_t)m * ldo + n);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (add)
            v[g][r] = (whole ? old[r] : p.out[(size_t)m * ldo + min(n + r, p.N - 1)]) + (v[g][r] + bias[g][r]);
          else if (p.flags & FLAG_GELU)
            v[g][r] = gelu_tanh_short(v[g][r] + bias[g][r]);
          else
            v[g][r] = activate<false>(p.flags & ~FLAG_GELU, v[g][r] + bias[g][r]);
        }
      }
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int n = nt + 8 * g;
        if (vec && n + 4 <= p.N) {
          *(f32x4_t*)(out + (size_t)m * ldo + n) = v[g];
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (n + r < p.N) out[(size_t)m * ldo + n + r] = v[g][r];
        }
      }
    }
  }
}

#define SKF_WAVES_FEW 8   // waves a block where the blocks are fewer than the compute units
#define SKF_WAVES_MANY 4  // and where every unit has a block or more (8: 12.1 us instead of 10.6 for 4,800 features of 1,600)
#define SKF_MAX_WAVES 8
#define SKF_MAX_ROWS 64
#define SKF_SPLIT_FROM 5000000L  // elements of a matrix from which a split of K pays
#define SKF_CHUNK 64                    // columns of a chunk
#define SKF_STRIDE (SKF_CHUNK + 4)      // floats between a chunk's rows in LDS: no two of a load's lanes share a bank

// Up to 64 rows, in RB blocks of 16.  A block owns 16 features and, where K is split over
// blockIdx.y, a run of chunks of 64 columns; its waves take the run's chunks in turn, each wave on
// its own (no barrier inside the loop).  A chunk of the weights comes from memory as 256
// contiguous bytes a feature, four features a load, goes through the wave's own piece of LDS and
// comes back in the layout of v_mfma_f32_16x16x4_f32: lane l holds columns 4 * (l / 16) .. + 3 of
// each 16 of feature l % 16.  The rows are the other operand, read in that layout from the L2,
// where they stay.  The next chunk is asked for before this one is multiplied; other waves cover
// the rest of the wait (a deeper queue was slower: 82 us against 72 for the vocabulary's matrix
// at 8 rows).  The same instructions run for every number of rows that fills the same blocks of
// 16, and a block of rows is multiplied on its own, so a row's result does not depend on the
// others.  With four blocks of rows the instructions bound the stream at some 4.8 TB/s.
template <int RB>
__global__ __launch_bounds__(64 * SKF_MAX_WAVES) void gemm_f32_skinny_kernel(GemmArgs p) {
  // (native vectors: a struct copied to LDS keeps what was loaded out of registers)
  __shared__ f32x4_t stage[SKF_MAX_WAVES][16 * SKF_STRIDE / 4];
  static_assert(sizeof(float) * SKF_MAX_WAVES * RB * 256 <= sizeof(f32x4_t) * SKF_MAX_WAVES * (16 * SKF_STRIDE / 4),
                "the waves' sums fit where the chunks were");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, n_waves = blockDim.x >> 6;
  const int n0 = blockIdx.x * 16;
  const int l16 = lane & 15, kq = lane >> 4;
  // features and rows that are not there read the last one that is; nothing of theirs is stored
  const float* wsrc[4];  // load i: feature 4 * i + l / 16, columns 4 * (l % 16) .. + 3 of the chunk
#pragma unroll
  for (int i = 0; i < 4; ++i) wsrc[i] = p.W + (size_t)min(n0 + 4 * i + kq, p.N - 1) * p.ldw;
  const float* arow[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b) arow[b] = p.A + (size_t)min(16 * b + l16, p.M - 1) * p.lda;
  f32x4_t* mine = stage[wave];
  const int n_chunks = (p.K + SKF_CHUNK - 1) / SKF_CHUNK;
  const int per_split = (n_chunks + p.n_splits - 1) / p.n_splits;
  const int c_end = min(n_chunks, (blockIdx.y + 1) * per_split);

  f32x4_t wv[4], av[RB][4];
  // columns beyond K (in the last chunk) and chunks beyond the run (asked for ahead by the wave's
  // last round) are read from inside the matrix; the rows' values beyond K count as zero
  auto ask = [&](int c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) wv[i] = *(const f32x4_t*)(wsrc[i] + min(c * SKF_CHUNK + 4 * l16, p.K - 4));
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
      for (int t = 0; t < 4; ++t)
        av[b][t] = *(const f32x4_t*)(arow[b] + min(c * SKF_CHUNK + 16 * t + 4 * kq, p.K - 4));
  };
  f32x4_t acc[RB];
#pragma unroll
  for (int b = 0; b < RB; ++b) acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  int c = blockIdx.y * per_split + wave;
  ask(c);
  for (; c < c_end; c += n_waves) {
    f32x4_t a[RB][4];
#pragma unroll
    for (int i = 0; i < 4; ++i) mine[(4 * i + kq) * (SKF_STRIDE / 4) + l16] = wv[i];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float live = c * SKF_CHUNK + 16 * t + 4 * kq < p.K ? 1.f : 0.f;
#pragma unroll
      for (int b = 0; b < RB; ++b) a[b][t] = av[b][t] * live;
    }
    ask(c + n_waves);
    __builtin_amdgcn_wave_barrier();  // (orders the compiler; a wave's LDS accesses run in order)
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const f32x4_t w = mine[l16 * (SKF_STRIDE / 4) + 4 * t + kq];
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[b][t].x, w.x, acc[b], 0, 0, 0);
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[b][t].y, w.y, acc[b], 0, 0, 0);
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[b][t].z, w.z, acc[b], 0, 0, 0);
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[b][t].w, w.w, acc[b], 0, 0, 0);
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  // accumulator r of lane l: row 4 * (l / 16) + r of its block of rows, feature l % 16.  The
  // waves' sums are added in the order of the waves, one thread an output and block of rows.
  __syncthreads();  // the pieces of LDS are no longer read
  float* parts = (float*)&stage[0][0];  // [wave][block of rows][row][feature]
#pragma unroll
  for (int b = 0; b < RB; ++b)
#pragma unroll
    for (int r = 0; r < 4; ++r) parts[((wave * RB + b) * 16 + 4 * kq + r) * 16 + l16] = acc[b][r];
  __syncthreads();
  if (tid < 256) {
    const int n = n0 + (tid & 15);
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const int m = 16 * b + (tid >> 4);
      if (m >= p.M || n >= p.N) continue;
      float v = parts[b * 256 + tid];
      for (int w = 1; w < n_waves; ++w) v += parts[(w * RB + b) * 256 + tid];
      if (p.n_splits > 1) {
        p.ws[((size_t)blockIdx.y * p.ws_rows + m) * p.N + n] = v;  // added up, and finished, by the caller's second kernel
        continue;
      }
      if (p.bias) v += p.bias[n];
      const size_t idx = (size_t)m * p.ldo + n;
      if (p.flags & FLAG_ACCUMULATE)
        p.out[idx] += v;
      else
        p.out[idx] = activate<false>(p.flags, v);
      if (p.k_pages && n >= p.q_width) *page_place(p, m, n) = v;
    }
  }
}

DEFINE_LAST_ERROR(mlxlm_last_error)

// What a tile shape costs in microseconds.  The 32-bit instructions' tiles: their products at the speed of a CU's matrix units (2.5e-4 an
// output and 64 columns, 8 % more in the smallest tiles, which read most, 3 % more in the largest; a block alone on its CU, one wave a
// SIMD, a fifth more), blocks that share a CU one after another, and a fixed part for the first step's way and the
// epilogue.  Against the times of 11 numbers of rows from 80 to 2,048 and ten matrices of widths 768 to 1,600, each with
// K in 1 to 8 parts, the choice is within 0.7 % of the best on average and 7 % at worst (1.7 % and 13 % with every tile
// at the same rate).
// Tiles of cut operands: `base` once, `tile` for each round of blocks that share a CU (`per_cu` of them), each 64 columns of K
// as many blocks as then share the CU (`chunk[0]` one, `chunk[1]` two, `chunk[2]` three), and the launch ahead that cuts the rows.  With them the choice among
// all shapes and parts is within 2.5 % of the best on average, for as many rows from 65 on and 15 matrices of widths 768 to 1,600.  (Prices fitted to today's
// kernels are within 1.1 %, but take K in fewer parts, longer sums: GPT-2 large, 1,050 tokens, logits off by 6.7e-7 instead of 6.1e-7.)
struct F32Price {
  int variant, bm, bn;
  double rate;  // (0: cut operands)
  int per_cu;
  double base, tile, chunk[3];
};
static const F32Price F32_PRICES[] = {{1, F32Tile64x128::BM, F32Tile64x128::BN, 1.03, 0, 0, 0, {}},
                                      {2, F32Tile64::BM, F32Tile64::BN, 1.0, 0, 0, 0, {}},
                                      {4, F32Tile32x64::BM, F32Tile32x64::BN, 1.08, 0, 0, 0, {}},
                                      {5, CutTile128::BM, CutTile128::BN, 0, 2, 0.0, 13.2, {1.53, 2.94, 0.0}},
                                      {6, CutTile64x128::BM, CutTile64x128::BN, 0, 2, 5.0, 6.3, {1.03, 1.91, 0.0}},
                                      {7, CutTile64::BM, CutTile64::BN, 0, 3, 5.7, 4.3, {0.69, 1.11, 1.6}}};
static inline bool is_cut(int variant) { return variant >= 5 && variant <= 7; }
static double price(const F32Price& s, int M, int N, int K, int n_splits) {
  const long tiles = (long)((M + s.bm - 1) / s.bm) * ((N + s.bn - 1) / s.bn);
  const int cus = n_compute_units(), chunks = ((K + 63) / 64 + n_splits - 1) / n_splits;
  // the busiest CU (of a die's run of tiles where operands are cut)
  const long n = is_cut(s.variant) ? ((tiles + N_DIES - 1) / N_DIES * n_splits + cus / N_DIES - 1) / (cus / N_DIES) : (tiles * n_splits + cus - 1) / cus;
  if (!is_cut(s.variant)) return 4.0 + (n == 1 ? 1.2 : 1.0) * n * chunks * (2.5e-4 * s.rate * s.bm * s.bn);
  const long full = n / s.per_cu, left = n % s.per_cu;
  return s.base + s.tile * (full + (left ? 1 : 0)) + chunks * (full * s.chunk[s.per_cu - 1] + (left ? s.chunk[left - 1] : 0.0)) +
         (2.3e-6 * M + 0.1e-6 * N) * K;
}
static int cheapest_shape(int M, int N, int K, int n_splits, double* us, bool cuts = true) {
  int variant = 0;
  for (const F32Price& s : F32_PRICES) {
    if (is_cut(s.variant) && (K < CUT_FROM_K || !cuts)) continue;
    const double t = price(s, M, N, K, n_splits) * (is_cut(s.variant) ? 1.04 : 1.0);  // (to be ahead for certain)
    if (!variant || t < *us) variant = s.variant, *us = t;
  }
  return variant;
}

// In how many parts K should go.  Up to 64 rows (the kernel for few rows): so that its blocks fill
// the GPU, one and a half blocks a compute unit, eight chunks of 64 columns a part at least; 1 where
// the matrix gives a block to every unit anyway, or is so small that a second kernel costs more
// than the split gains.  More rows: by the prices above and the second kernel's, a launch plus the
// bytes of the partial sums at 3 TB/s.  `fused`: it stands in for one that would run anyway (the norm
// that follows a sum into the residual stream), so it costs only the extra bytes.
extern "C" int gemm_f32_splits(int M, int N, int K, int fused, int force) {
  const int n_chunks = (K + SKF_CHUNK - 1) / SKF_CHUNK;
  if (M < 1) return 1;
  int want;
  if (force > 0) {
    want = force;
  } else if (M <= SKF_MAX_ROWS) {
    const int n_blocks = (N + 15) / 16;
    if (n_blocks >= n_compute_units() || (long)N * K < SKF_SPLIT_FROM) return 1;
    want = (3 * n_compute_units() / 2 + n_blocks - 1) / n_blocks;
    if (want > n_chunks / 8) want = n_chunks / 8;
  } else {
    double best_us = 0.0;
    want = 1;
    for (int s = 1; s <= 8 && s <= n_chunks / 2; ++s) {
      double us = 0.0;
      cheapest_shape(M, N, K, s, &us);
      if (s > 1) us += (fused ? 1.0 : 2.5) + 8.0 * (fused ? s - 1 : s) * (double)M * N / 3e6;
      if (s == 1 || us < 0.99 * best_us) want = s, best_us = us;
    }
  }
  if (want < 1) want = 1;
  if (want > n_chunks) want = n_chunks;
  const int per = (n_chunks + want - 1) / want;
  return (n_chunks + per - 1) / per;  // no empty part
}

template <typename S>
static void launch_tiles(const GemmArgs& p, hipStream_t stream) {
  dim3 grid((p.N + S::BN - 1) / S::BN, (p.M + S::BM - 1) / S::BM, p.n_splits), block(S::THREADS);
  hipLaunchKernelGGL(gemm_f32_tile_kernel<S>, grid, block, 0, stream, p);
}
template <typename S>
static void launch_cut_tiles(const GemmArgs& p, hipStream_t stream) {
  const long tiles = (long)((p.M + S::BM - 1) / S::BM) * ((p.N + S::BN - 1) / S::BN);
  dim3 grid((unsigned)((tiles + N_DIES - 1) / N_DIES * N_DIES), p.n_splits), block(S::THREADS);  // a run of tiles for each die
  hipLaunchKernelGGL(gemm_f32_cut_kernel<S>, grid, block, 0, stream, p);
}

static void launch(const GemmArgs& p, int variant, hipStream_t stream) {
  if (variant == 1) return launch_tiles<F32Tile64x128>(p, stream);
  if (variant == 2) return launch_tiles<F32Tile64>(p, stream);
  if (variant == 4) return launch_tiles<F32Tile32x64>(p, stream);
  if (variant == 5) return launch_cut_tiles<CutTile128>(p, stream);
  if (variant == 6) return launch_cut_tiles<CutTile64x128>(p, stream);
  if (variant == 7) return launch_cut_tiles<CutTile64>(p, stream);
  // where the blocks are fewer than the compute units, more waves each
  const int blocks = (p.N + 15) / 16;
  const int waves = blocks * p.n_splits < n_compute_units() ? SKF_WAVES_FEW : SKF_WAVES_MANY;
  const dim3 grid(blocks, p.n_splits), block(64 * waves);
  if (p.M <= 16)
    hipLaunchKernelGGL(gemm_f32_skinny_kernel<1>, grid, block, 0, stream, p);
  else if (p.M <= 32)
    hipLaunchKernelGGL(gemm_f32_skinny_kernel<2>, grid, block, 0, stream, p);
  else if (p.M <= 48)
    hipLaunchKernelGGL(gemm_f32_skinny_kernel<3>, grid, block, 0, stream, p);
  else
    hipLaunchKernelGGL(gemm_f32_skinny_kernel<4>, grid, block, 0, stream, p);
}

// 1 if gemm_f32_scatter puts the keys and values of so many rows into their pages.  (Up to 64 rows: a step of GPT-2 large at 30 to
// 60 keys without the 36 launches that did it, 1 / 8 / 16 / 17 / 32 / 64 rows, 1,705 -> 1,595, 1,909 -> 1,800, 2,190 -> 2,072, 2,362 ->
// 2,283, 2,850 -> 2,744, 4,585 -> 4,534 us; of small with 12, 514 -> 492 to 1,361 -> 1,350.  A tile's epilogue does not: its pieces of 16 bytes a
// row, each at a place of its own, cost more than the launch that writes whole heads, 15,002 -> 15,122 us for 1,050 rows.)
extern "C" int gemm_f32_scatters(int M, int n_splits) { return M >= 1 && M <= SKF_MAX_ROWS && n_splits == 1; }

static inline int cut_stride(int K) { return (K + 31) / 32 * 32; }
static inline bool fits_tiles(int lda, int ldw, int K, bool cut) {
  return (cut ? fits_copy_buffer((size_t)128 * cut_stride(K) * 4) : fits_copy_buffer(((size_t)127 * lda + K) * 4)) &&
         fits_copy_buffer(((size_t)127 * ldw + K) * 4);
}
static int choose(int M, int N, int K, int variant, int n_splits, bool cuts = true) {
  double us = 0.0;
  return variant != 0 ? variant : M <= SKF_MAX_ROWS ? 3 : cheapest_shape(M, N, K, n_splits, &us, cuts);
}
// Rows that are cut at once: up to 256 MB of them (a prompt of 8,192 rows of 6,400 has 210), so that the room does not grow with the
// rows and a grid of one block a row and feature holds them.
static inline int cut_at_once(int M, int K) {
  const int most = ((64 << 20) / cut_stride(K) + 127) / 128 * 128;
  return M < most ? M : most;
}
#define CUT_BLOCKS (1 << 23)  // features whose scales a launch finds at most (a grid holds less than 2^32 threads)
// Floats of memory that gemm_f32_scatter needs for a product of these sizes: as many rows as are cut at once, and a scale a row and
// feature (0: tiles of cut operands don't take it).
extern "C" size_t gemm_f32_room(int M, int N, int K, int variant, int n_splits) {
  if (M <= 0 || !is_cut(choose(M, N, K, variant, n_splits))) return 0;
  const size_t rows = cut_at_once(M, K);
  return rows * cut_stride(K) + 2 * (rows + N);
}

// variant: 0 = choose, 1 = tiles of 64 x 128, 2 = of 64 x 64, 4 = of 32 x 64, 3 = the kernel for up to
// 64 rows, 5 = tiles of cut operands of 128 x 128, 6 = of 64 x 128, 7 = of 64 x 64.  n_splits > 1: K in that many parts, whose sums go to ws[part][M][N] (ws_floats floats at least) for sum_partials of gemm_bf16_decode.hip to add up
// and finish; out is not written then.
// k_pages: the features from q_width on go to the pages of the key/value cache too (mlx_lm/models/cache.py:352-354).
extern "C" int gemm_f32_scatter(void* out, const void* A, const void* W, const float* bias, int M, int N,
                                int K, int lda, int ldw, int ldo, int flags, int variant, int n_splits, float* ws,
                                size_t ws_floats, void* k_pages, void* v_pages, size_t page_stride, const int* block_table,
                                int max_blocks, const int* token_req, const int* positions, int q_width, int kv_width,
                                int head_dim, int page_size, float* room, size_t room_floats, hipStream_t stream) {
  GemmArgs p = {};
  p.A = (const float*)A;
  p.W = (const float*)W;
  p.bias = bias;
  p.out = (float*)out;
  p.M = M, p.N = N, p.K = K, p.ws_rows = M;
  p.lda = lda, p.ldw = ldw, p.ldo = ldo;
  p.flags = flags;
  p.n_splits = 1, p.per_split = (K + SKF_CHUNK - 1) / SKF_CHUNK, p.ws = nullptr;
  if (M < 0 || N <= 0 || K <= 0) FAIL("gemm_f32: bad sizes M=%d N=%d K=%d", M, N, K);
  if (K % 4 != 0) FAIL("gemm_f32: K=%d must be a multiple of 4", K);
  if (lda % 4 != 0 || ldw % 4 != 0)
    FAIL("gemm_f32: row strides lda=%d ldw=%d must be multiples of 4", lda, ldw);
  if (lda < K || ldw < K || ldo < N)
    FAIL("gemm_f32: row strides smaller than the rows (lda=%d ldw=%d ldo=%d)", lda, ldw, ldo);
  if (!A || !W || !out) FAIL("gemm_f32: null pointer");
  if (((uintptr_t)A | (uintptr_t)W) & 15) FAIL("gemm_f32: A and W must be 16-byte aligned");
  if ((flags & FLAG_ACCUMULATE) && (flags & FLAG_ACT_ANY))
    FAIL("gemm_f32: an activation and accumulate cannot be combined");
  if (M == 0) return 0;
  if (n_splits < 1) FAIL("gemm_f32: n_splits=%d", n_splits);
  if (n_splits > 1) {
    const int n_chunks = (K + SKF_CHUNK - 1) / SKF_CHUNK, per = (n_chunks + n_splits - 1) / n_splits;
    if (n_splits > n_chunks) FAIL("gemm_f32: %d parts of K=%d", n_splits, K);
    if (!ws || ws_floats < (size_t)n_splits * M * N) FAIL("gemm_f32: the parts' workspace is too small");
    p.n_splits = n_splits, p.per_split = per, p.ws = ws;
  }
  if (k_pages) {
    if (!gemm_f32_scatters(M, n_splits) || (variant != 0 && variant != 3) || (flags & (FLAG_ACCUMULATE | FLAG_ACT_ANY)))
      FAIL("gemm_f32: the cache scatter is the kernel for few rows', with a plain epilogue and K whole");
    if (!v_pages || !block_table || !token_req || !positions || head_dim <= 0 || page_size <= 0 || max_blocks <= 0 ||
        kv_width % head_dim != 0 || q_width + 2 * kv_width != N)
      FAIL("gemm_f32: the cache scatter's pointers or widths (q_width %d + 2 * kv_width %d, N=%d)", q_width, kv_width, N);
    if (head_dim < 4 || head_dim > 256 || head_dim % 4 != 0 || page_stride < (size_t)kv_width * page_size)  // (as kv_write has it)
      FAIL("gemm_f32: heads of %d, or a page stride smaller than a page", head_dim);
    p.k_pages = (float*)k_pages, p.v_pages = (float*)v_pages, p.page_stride = page_stride;
    p.block_table = block_table, p.max_blocks = max_blocks, p.token_req = token_req, p.positions = positions;
    p.q_width = q_width, p.kv_width = kv_width, p.head_dim = head_dim, p.page_size = page_size;
  }
  variant = choose(M, N, K, variant, n_splits, room != nullptr);  // (0 without room: not those that need it)
  if (variant != 3 && p.per_split * (n_splits - 1) * SKF_CHUNK >= K) FAIL("gemm_f32: %d parts of K=%d leave one empty", n_splits, K);
  if (variant == 3 && M > SKF_MAX_ROWS)
    FAIL("gemm_f32: the kernel for few rows takes at most %d, got %d", SKF_MAX_ROWS, M);
  if (variant < 1 || variant > 7) FAIL("gemm_f32: unknown variant %d", variant);
  const size_t room_wanted = gemm_f32_room(M, N, K, variant, n_splits);
  // Rows some 8 million floats apart or more are beyond the 32-bit offsets of a tile's copies: the kernel for few
  // rows, which has pointers, takes them 64 at a time.  More tiles of rows than a grid holds go in several launches.
  if (!fits_tiles(lda, ldw, K, is_cut(variant))) variant = 3;
  if (is_cut(variant)) {
    if (!room || ((uintptr_t)room & 15) || room_floats < room_wanted)
      FAIL("gemm_f32: tiles of cut operands need %zu floats of aligned memory", room_wanted);
    const int rows = cut_at_once(M, K);
    RowScale* const scales = (RowScale*)(room + (size_t)rows * cut_stride(K));
    p.cut = room, p.ldc = cut_stride(K), p.a_scales = scales, p.w_scales = scales + rows;
    for (int m = 0; m < M; m += rows) {
      p.M = M - m < rows ? M - m : rows;
      // (the features' scales lie behind those of the first rows, which are as many as any that follow)
      CutArgs c = {p.A, p.W, p.M, m ? 0 : N < CUT_BLOCKS ? N : CUT_BLOCKS, K, lda, ldw, p.ldc, (u32x4_t*)room, scales};
      hipLaunchKernelGGL(cut_rows_kernel, dim3((unsigned)(c.M + (c.N + 3) / 4)), dim3(256), 0, stream, c);
      for (int n = c.N; m == 0 && n < N; n += c.N) {
        c.M = 0, c.N = N - n < CUT_BLOCKS ? N - n : CUT_BLOCKS, c.W = p.W + (size_t)n * ldw, c.scales = scales + rows + n;
        hipLaunchKernelGGL(cut_rows_kernel, dim3((unsigned)((c.N + 3) / 4)), dim3(256), 0, stream, c);
      }
      launch(p, variant, stream);
      p.A += (size_t)p.M * lda, p.out += (size_t)p.M * ldo;
      if (n_splits > 1) p.ws += (size_t)p.M * N;
    }
    CHECK_LAUNCH("gemm_f32");
    return 0;
  }
  const int most = variant == 3 ? SKF_MAX_ROWS : 65535 * (variant == 4 ? F32Tile32x64::BM : F32Tile64::BM);
  static_assert(F32Tile64x128::BM == F32Tile64::BM, "both tiles' rows");
  for (int left = M; left > 0; left -= most) {
    p.M = left < most ? left : most;
    p.through = fits_through_buffer((size_t)p.M * (n_splits > 1 ? N : ldo) * 4);
    launch(p, variant, stream);
    p.A += (size_t)most * lda, p.out += (size_t)most * ldo;
    if (p.ws) p.ws += (size_t)most * N;
  }
  CHECK_LAUNCH("gemm_f32");
  return 0;
}
