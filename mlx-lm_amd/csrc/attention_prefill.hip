// Prefill attention for bfloat16 caches on the matrix cores: portions of
// prompts, 128 consecutive queries of one request per block, keys and values
// read from the pages in tiles of 64.  Same contract as attn_tile in
// attention.hip (same tile list, with up to 128 rows a tile); this is the
// kernel that serving uses for head sizes 32, 64, 128 and 256, attn_tile stays as
// the general one (any head size, float caches).
//
// Replaces scaled_dot_product_attention with the "causal" mask and a cache
// offset (mlx_lm/models/base.py:24-35,132-139, mlx_lm/models/gpt2.py:60-65).
//
// Data flow, chosen so that a lane only ever deals with one query:
//  * Each of the four waves owns 32 queries.  Scores are computed transposed,
//    S^T = K Q^T, with v_mfma_f32_32x32x16_bf16: keys are the rows (A-operand,
//    from LDS), the wave's queries the columns (B-operand, kept in registers).
//    A lane then holds 16 scores of query (lane % 32) per 32-key subtile, so
//    the row maximum and sum need a single cross-lane step.
//  * The rows of a subtile are fed in a permuted key order such that the 8
//    scores a lane holds per 16-key chunk are 8 *consecutive* keys.  They are
//    exactly the B-operand fragment of O^T = V^T P^T; no shuffle, no LDS.
//  * V^T is needed with keys contiguous.  Values sit in the pages with head
//    columns contiguous, so the value tile is transposed on its way into LDS:
//    a thread reads the same 8 columns of two neighbouring keys and writes
//    eight 32-bit words (two keys each).
//  * Online softmax in 32-bit per lane; outputs leave as O^T accumulators.
// Heads of 64 without optional terms of a score have a kernel of their own, attn_prefill_ring_kernel, with the same
// products and the same softmax: tiles go into LDS as they lie in the pages, by copies, and the values are transposed
// on their way out of it.
// What bounds it: the softmax's vector instructions (here some 1,150 cycles of them a wave and tile of 64 keys beside 512 of
// the matrix unit, a third of them addresses and the values' transposition), and at few blocks the chain of one block.
// 2 x 1,024 tokens of 16 heads of 128: 34.6 us; of 8 heads of 256: 100 (107 with two tiles on their way, which did not fit
// the registers).
#include "common.h"
#include "attention_tiles.h"
#include "attention_decode_row.h"
#include "lds_copy.h"
#include <type_traits>

struct PrefillArgs {
  uint16_t* out;
  int out_by_16;  // a head's row of out is whole pieces of 16 bytes
  const uint16_t* q;
  const uint16_t* k_pages;
  const uint16_t* v_pages;
  const int* block_table;
  const int* token_req;
  const int* positions;
  const int* tiles;  // (first row, n rows <= 128) pairs
  size_t page_stride;
  int ldq, ldo, max_blocks;
  int n_heads, n_kv_heads, page_size, window;
  int page_shift;  // log2(page_size), or -1 if that is no power of two
  float scale;
  // Optional terms (the kernel's EXTRAS variant; all absent: plain causal attention), as in
  // attention.hip's AttnArgs: head_scale [n_heads] instead of `scale`; slopes [n_heads], slope *
  // distance taken off a score; keep_first, the first keys that a window leaves visible; gate
  // (bfloat16 rows of stride ldg), the output times its sigmoid.
  const float* head_scale;
  const float* slopes;
  const uint16_t* gate;
  int ldg, keep_first;
  // softcap > 0: a scaled score s becomes softcap * tanh(s / softcap); dist_bias [n_heads, n_dist]:
  // dist_bias[h][min(distance, n_dist - 1)] is added to a score (the kernel's SHAPED variant)
  float softcap;
  const float* dist_bias;
  int n_dist;
  // sinks [n_heads]: exp(sinks[h]) in the softmax's denominator; head_gate (rows of stride ldhg): head
  // h's output times the sigmoid of column h
  const float* sinks;
  const float* head_gate;
  int ldhg;
};

#define BQ ATTN_PREFILL_TILE_QUERIES  // queries per block
#define KT 64   // keys per tile
#define VT_STRIDE (KT + 8)  // 144 bytes a row: 16-byte reads of 32 rows fall on distinct banks

union Frag8 {
  uint4 u;
  bf16x8_t v;
};

// S^T row rho of a 32-key subtile holds this key of the subtile (see above)
__device__ __forceinline__ int key_of_row(int rho) {
  const int j = rho >> 3, g = (rho >> 2) & 1, i = rho & 3;
  return 16 * (j >> 1) + 8 * g + 4 * (j & 1) + i;
}

// POW2: the page size is a power of two (a key's page and row are a shift and a mask)
// EXTRAS: the optional terms of PrefillArgs are looked at (the plain variant has no trace of them)
// SHAPED (with EXTRAS): scores also pass the soft cap and take the distance table's term
// GROUPS: groups of four waves, which take the key tiles by turns, each group with LDS of its own, and join their sums at
// the end.  A block's walk over its keys is one tile after another (copy, barrier, products, softmax: some 1.2 us), and
// where the blocks are few the longest walk is the kernel's time: two groups halve it.  A walk of fewer than
// TWO_GROUPS_FROM tiles is left to the first group: joining the sums costs about as much as a tile (25 heads of 64, both
// groups and the first alone: 17 tokens, one tile, 5.3 and 4.5 us; 192, three, 8.6 and 7.7; 300, five, 10.1 and 9.5; 333,
// six, 10.6 and 10.9; 333 under a window of 200, six at most, 11.7 and 13.1.  16 heads of 32: 192 tokens 6.4 and 5.9; 200,
// four tiles, 6.5 and 7.2; the kernel for heads of 64 without terms, five tiles 10.1 and 9.8, six 9.3 and 9.6.)  That the
// other waves were there at all costs up to 0.4 us (128 tokens: 7.0, in a block of four
// waves 6.8), but how long the walks are is not known where the kernel is launched: a recorded step runs at other lengths.
// (With heads of 64 two waves a SIMD, no fewer and no more, are named to the compiler: left alone it takes the registers
// of three, which leaves it less to overlap.  Heads of 32 run three where blocks are many: 16 heads at
// 8,000 tokens 133 us, 141 with two.)
template <int HD>
static constexpr int TWO_GROUPS_FROM = HD == 32 ? 4 : 6;
template <int HD, bool POW2, bool EXTRAS, bool SHAPED, int GROUPS>
__global__ __launch_bounds__(256 * GROUPS) __attribute__((amdgpu_waves_per_eu(HD <= 64 ? 2 : 1, HD == 32 ? 8 : HD == 64 ? 2 : 1)))
void attn_prefill_kernel(PrefillArgs p) {
  constexpr int KS_STRIDE = HD + 8;
  constexpr int DC = HD / 16;           // 16-column chunks of a head (QK contraction steps)
  constexpr int DT = HD / 32;           // 32-row tiles of O^T
  constexpr int K_CHUNKS = KT * HD / 8; // 16-byte pieces of a key tile
  constexpr int K_PER_T = (K_CHUNKS + 255) / 256;
  constexpr int V_ITEMS = (KT / 2) * (HD / 8);  // (key pair, 8-column chunk) items of a value tile
  constexpr int V_PER_T = (V_ITEMS + 255) / 256;
  // tiles on their way: two, or one where a tile is so many registers that two would not fit (heads of 256)
  constexpr int SETS = HD <= 128 ? 2 : 1, SECOND = SETS - 1;
  constexpr int GROUP_LDS = KT * KS_STRIDE + HD * VT_STRIDE;
  __shared__ __attribute__((aligned(16))) uint16_t tiles_lds[GROUPS * GROUP_LDS];

  const int group = GROUPS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
  const int tid = threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;  // (within the group)
  uint16_t* const Ks = tiles_lds + group * GROUP_LDS;
  uint16_t* const Vt = Ks + KT * KS_STRIDE;
  // Which tile and head.  The tiles come with the most keys first, and a tile's heads are
  // neighbours in the launch, so the blocks with the longest walks start first and the short
  // ones fill in behind them (with the tiles as the fast index, a CU's two blocks were two
  // equally long ones, which took turns on its SIMDs to the end: 32 us a layer instead of 26
  // for 2 x 1,024 tokens of GPT-2 XL).
  const int h = blockIdx.x, tile = blockIdx.y;
  const int row0 = p.tiles[2 * tile];
  const int nq = p.tiles[2 * tile + 1];
  const int kv_head = h / (p.n_heads / p.n_kv_heads);
  const int pos0 = p.positions[row0];
  const int* table = p.block_table + (size_t)p.token_req[row0] * p.max_blocks;
  const uint32_t head_off = (uint32_t)(kv_head * p.page_size * HD);  // (within a page: below its stride)

  const int ql = lane & 31, g = lane >> 5;
  const int qi = wave * 32 + ql;         // this lane's query within the tile
  const bool q_live = qi < nq;
  const int qpos = pos0 + qi;
  const int q_lo = p.window > 0 ? max(0, qpos - p.window + 1) : 0;

  // the wave's queries as B-operand fragments: column = query, k = head columns
  Frag8 qf[DC];
  {
    const uint16_t* qrow = p.q + (size_t)(row0 + min(qi, nq - 1)) * p.ldq + h * HD + 8 * g;
#pragma unroll
    for (int dc = 0; dc < DC; ++dc) {
      const uint4 t = *(const uint4*)(qrow + dc * 16);
      qf[dc].u = q_live ? t : make_uint4(0u, 0u, 0u, 0u);
    }
  }

  const int k_hi = pos0 + nq;  // one past the last key any query of the tile sees
  const int k_lo = p.window > 0 ? max(0, pos0 - p.window + 1) : 0;
  const int kt0 = (k_lo / KT) * KT;
  // keys this wave's queries can see end here; later tiles it only helps to load
  const int wave_hi = min(k_hi, pos0 + wave * 32 + 32);
  const int wave_q0 = pos0 + wave * 32;            // position of the wave's first query
  const float c2 = (EXTRAS && p.head_scale ? p.head_scale[h] : p.scale) * 1.4426950408889634f;  // scores to units of log 2
  const float slope2 = EXTRAS && p.slopes ? p.slopes[h] * 1.4426950408889634f : 0.f;
  // the kept first keys [0, sink_hi) that the tile's window has left behind: tiles of their own, first
  const int sink_hi = EXTRAS ? min(p.window > 0 ? p.keep_first : 0, k_lo) : 0;
  const int n_sink_tiles = (sink_hi + KT - 1) / KT;
  const int n_sink_pages = sink_hi > 0 ? (sink_hi - 1) / p.page_size + 1 : 0;
  // (in a short walk the second group's waves end here: barriers count the waves that are left)
  const int groups = GROUPS > 1 && n_sink_tiles + (k_hi - kt0 + KT - 1) / KT >= TWO_GROUPS_FROM<HD> ? GROUPS : 1;
  if (GROUPS > 1 && group >= groups) return;

  float m = -INFINITY, l = 0.f;
  f32x16_t ot[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) ot[dt][r] = 0.f;

  // (the keys' two sets as arrays of their own: as one array indexed by the set they stayed in
  // scratch memory)
  uint4 kreg0[K_PER_T], kreg1[K_PER_T], vreg[SETS][V_PER_T][2];

  // The request's page numbers go to LDS once: a load of keys or values then
  // depends on no other load from memory, and two tiles can be on their way
  // while one is multiplied.  (Looked up from memory per load, every load
  // waited for its page number first: eight trips to memory in a row per tile.)
  extern __shared__ int page_of[];  // [max_blocks]
  const int pg0 = k_lo / p.page_size;
  const int n_pg = (k_hi - 1) / p.page_size - pg0 + 1;
  for (int i = threadIdx.x; i < n_sink_pages; i += 256 * groups) page_of[i] = table[i];
  for (int i = threadIdx.x; i < n_pg; i += 256 * groups) page_of[n_sink_pages + i] = table[pg0 + i];
  __syncthreads();

  // Loads are never predicated and never zeroed: a key outside [k_lo, k_hi) is
  // read from the nearest key inside (a valid address with finite numbers);
  // its score is masked below, so its probability is zero.
  // An address is a dozen integer instructions, four times a thread and tile, in a kernel whose
  // time is its vector instructions: a division by a run-time page size alone costs thirty, and
  // choosing between it and a shift at run time put a branch around every address.  So the
  // choice is the kernel's template argument, and everything but the page's start is 32-bit.
  const uint32_t stride32 = (uint32_t)p.page_stride;
  const int shift = p.page_shift, row_mask = p.page_size - 1;
  // (a tile's first key says of which run it is: at or beyond 2^29, the kept first keys')
  constexpr int SINK = 1 << 29;
  auto address = [&](int key, int col) __attribute__((always_inline)) -> size_t {
    int kk = min(max(key, k_lo), k_hi - 1);
    int first_page = pg0 - n_sink_pages;
    if (EXTRAS && key >= SINK) kk = min(key - SINK, sink_hi - 1), first_page = 0;
    int idx, row;
    if constexpr (POW2) {
      idx = kk >> shift, row = kk & row_mask;
    } else {
      idx = kk / p.page_size, row = kk - idx * p.page_size;
    }
    const uint32_t within = head_off + (uint32_t)(row * HD + col);
    return (size_t)(uint32_t)page_of[idx - first_page] * stride32 + within;
  };
  auto fetch = [&](int kt, const int set) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < K_PER_T; ++i) {
      const int c = min(tid + 256 * i, K_CHUNKS - 1);  // surplus threads repeat the last piece
      const uint4 t = *(const uint4*)(p.k_pages + address(kt + c / (HD / 8), (c % (HD / 8)) * 8));
      if (set == 0) kreg0[i] = t; else kreg1[i] = t;
    }
#pragma unroll
    for (int i = 0; i < V_PER_T; ++i) {
      const int it = min(tid + 256 * i, V_ITEMS - 1);
      const int jp = it % (KT / 2), col = (it / (KT / 2)) * 8;
#pragma unroll
      for (int e = 0; e < 2; ++e) vreg[set][i][e] = *(const uint4*)(p.v_pages + address(kt + 2 * jp + e, col));
    }
  };
  auto stage = [&](const int set) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < K_PER_T; ++i) {
      const int c = tid + 256 * i;
      if (K_CHUNKS % 256 == 0 || c < K_CHUNKS)
        *(uint4*)(Ks + (c / (HD / 8)) * KS_STRIDE + (c % (HD / 8)) * 8) = set == 0 ? kreg0[i] : kreg1[i];
    }
#pragma unroll
    for (int i = 0; i < V_PER_T; ++i) {
      const int it = tid + 256 * i;
      if (V_ITEMS % 256 == 0 || it < V_ITEMS) {
        const int jp = it % (KT / 2), col = (it / (KT / 2)) * 8;
        const uint32_t a[4] = {vreg[set][i][0].x, vreg[set][i][0].y, vreg[set][i][0].z, vreg[set][i][0].w};
        const uint32_t b[4] = {vreg[set][i][1].x, vreg[set][i][1].y, vreg[set][i][1].z, vreg[set][i][1].w};
        uint32_t* dst = (uint32_t*)(Vt + col * VT_STRIDE + 2 * jp);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          // columns col+2w and col+2w+1 of keys 2jp (low half) and 2jp+1 (high half)
          dst[(2 * w) * (VT_STRIDE / 2)] = (a[w] & 0xffffu) | (b[w] << 16);
          dst[(2 * w + 1) * (VT_STRIDE / 2)] = (a[w] >> 16) | (b[w] & 0xffff0000u);
        }
      }
    }
  };

  // One tile: its keys and values go from registers to LDS, the registers take
  // a later tile, then the arithmetic.
  // `steady` (a compile-time flag): the tile lies below every query of the block
  // and there is no window, so no wave is idle and nothing is masked; a loop of
  // such tiles has no branch inside, and the compiler lets the loads of the
  // other register set stay in flight while this one is staged.
  // `kt_next`: the first key of the tile whose loads start here, SETS tiles on.
  auto one_tile = [&](int kt_in, int kt_next, const int set, auto steady) __attribute__((always_inline)) {
    constexpr bool STEADY = decltype(steady)::value;
    __syncthreads();  // the previous tile is no longer read
    stage(set);
    __syncthreads();
    fetch(kt_next, set);  // (beyond the last tile: harmless reads of the last key)
    const bool sink = EXTRAS && kt_in >= SINK;
    const int kt = sink ? kt_in - SINK : kt_in;
    if constexpr (!STEADY) {
      if ((!sink && kt >= wave_hi) || wave * 32 >= nq) return;  // nothing here for this wave (uniform)
    }

    // ---- S^T = K Q^T for the two 32-key subtiles --------------------------------
    f32x16_t st[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int r = 0; r < 16; ++r) st[s][r] = 0.f;
      const uint16_t* krow = Ks + (32 * s + key_of_row(ql)) * KS_STRIDE + 8 * g;
#pragma unroll
      for (int dc = 0; dc < DC; ++dc) {
        Frag8 a;
        a.u = *(const uint4*)(krow + dc * 16);
        st[s] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, qf[dc].v, st[s], 0, 0, 0);
      }
    }
    // element r of subtile s: key kt + 32 s + 16 (r / 8) + 8 g + r % 8.
    // Scores are kept in units of log 2 (scale * log2(e) folded into one
    // factor), so that a probability is one fused multiply-add and one
    // v_exp_f32.  Tiles that every query of the wave sees whole (below the
    // diagonal, inside the window) skip the masks: this arithmetic, not the
    // MFMAs, is what the kernel's time goes to.
    const bool whole = STEADY || (!EXTRAS && kt + KT - 1 <= wave_q0 && (p.window <= 0 || kt >= wave_q0 + 31 - p.window + 1));
    float tmax = -INFINITY;
    if constexpr (EXTRAS) {
      // Scores in units of log 2 with the distance's share taken off: element r of subtile s is
      // the key kt + 8 g + off(s, r) with off a constant of the element, so the share is
      // slope2 * (off - (qpos - kt - 8 g)), one multiply-add on top of the score's own.
      const float far = slope2 * (float)(qpos - kt - 8 * g);
      // A tile that every query of the wave sees whole (below the diagonal and inside the window,
      // or all of it kept first keys) needs no masks.
      const bool all_seen = sink ? kt + KT <= sink_hi
                                 : (kt >= k_lo && kt + KT - 1 <= wave_q0 && wave_q0 + 31 < nq + pos0 &&
                                    (p.window <= 0 || kt >= wave_q0 + 31 - p.window + 1));
      if constexpr (SHAPED) {
        // the score in its own units first: the cap and the table's term are no linear function
        // of it.  tanh(x) = 1 - 2 / (exp(2 x) + 1) through the hardware's exp2 and reciprocal (an
        // exp2 that overflows gives the cap itself); a tile that lies wholly beyond the table's
        // reach takes the table's last entry without a look-up.
        const int run_lo = sink ? 0 : k_lo, run_hi = sink ? sink_hi : k_hi;
        const float c1 = p.head_scale ? p.head_scale[h] : p.scale;
        const float cap = p.softcap, cap_exp = cap > 0.f ? 2.0f * 1.4426950408889634f / cap : 0.f;
        const float* bias_row = p.dist_bias ? p.dist_bias + (size_t)h * p.n_dist : nullptr;
        const int last = p.n_dist - 1;
        const bool beyond = bias_row && wave_q0 - (kt + KT - 1) >= last;
        const float beyond_bias = beyond ? bias_row[last] : 0.f;
        const float raw_exp = c1 * cap_exp, cap2 = cap * 1.4426950408889634f;  // (the cap in units of log 2)
        auto shaped = [&](float raw, int o, int key) {
          const float away = fmaf(slope2, (float)o, -far);
          if (cap > 0.f && !bias_row)  // cap2 * tanh = cap2 - 2 cap2 / (exp + 1)
            return fmaf(__builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(raw * raw_exp) + 1.0f), -2.0f * cap2, cap2 + away);
          float v = raw * c1;
          if (cap > 0.f) v = cap * (1.0f - 2.0f * __builtin_amdgcn_rcpf(__builtin_amdgcn_exp2f(v * cap_exp) + 1.0f));
          if (beyond)
            v += beyond_bias;
          else if (bias_row)
            v += bias_row[min(max(qpos - key, 0), last)];
          return fmaf(v, 1.4426950408889634f, away);
        };
        if (all_seen) {
#pragma unroll
          for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const int o = 32 * s + 16 * (r >> 3) + (r & 7);
              st[s][r] = shaped(st[s][r], o, kt + 8 * g + o);
              tmax = fmaxf(tmax, st[s][r]);
            }
        } else {
#pragma unroll
          for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const int o = 32 * s + 16 * (r >> 3) + (r & 7);
              const int key = kt + 8 * g + o;
              const bool ok = q_live && key <= qpos && key >= run_lo && key < run_hi && (key >= q_lo || key < p.keep_first);
              st[s][r] = ok ? shaped(st[s][r], o, key) : -INFINITY;
              tmax = fmaxf(tmax, st[s][r]);
            }
        }
      } else if (all_seen) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float off = (float)(32 * s + 16 * (r >> 3) + (r & 7));
            st[s][r] = fmaf(st[s][r], c2, fmaf(slope2, off, -far));
            tmax = fmaxf(tmax, st[s][r]);
          }
      } else {
        // a key counts if it is of this tile's run and the query sees it (inside its window, or
        // one of the kept first)
        const int run_lo = sink ? 0 : k_lo, run_hi = sink ? sink_hi : k_hi;
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int o = 32 * s + 16 * (r >> 3) + (r & 7);
            const int key = kt + 8 * g + o;
            const bool ok = q_live && key <= qpos && key >= run_lo && key < run_hi && (key >= q_lo || key < p.keep_first);
            const float v = fmaf(st[s][r], c2, fmaf(slope2, (float)o, -far));
            st[s][r] = ok ? v : -INFINITY;
            tmax = fmaxf(tmax, st[s][r]);
          }
      }
    } else if (whole) {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int r = 0; r < 16; ++r) tmax = fmaxf(tmax, st[s][r]);
      tmax *= c2;  // c2 > 0: the largest score stays the largest
    } else {
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = kt + 32 * s + 16 * (r >> 3) + 8 * g + (r & 7);
          const bool ok = q_live && key <= qpos && key >= q_lo;
          st[s][r] = ok ? st[s][r] : -INFINITY;
          tmax = fmaxf(tmax, st[s][r] * c2);
        }
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, WAVE));
    // Probabilities are taken against the largest score so far: the weight that counts most is then exactly 1, which
    // the rounding to bfloat16 leaves as it is.  (Against a reference that lagged by up to 2^8 it was rounded like the
    // others while the sum took it unrounded: 25 heads of 64 at 8,000 tokens in 294 us instead of 309, but with sharp scores the
    // outputs were 10 to 30 % further from 64 bits.)
    if (__any(tmax > m)) {
      const float m_new = fmaxf(m, tmax);
      const float alpha = exp2f(m - (m_new == -INFINITY ? 0.f : m_new));  // (a row with no key yet: zero)
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) ot[dt][r] *= alpha;
      m = m_new;
    }
    const float m_use = (m == -INFINITY) ? 0.f : m;
    float lsum = 0.f;
    Frag8 pf[2][2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        float e[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          e[i] = EXTRAS ? __builtin_amdgcn_exp2f(st[s][8 * c + i] - m_use)
                        : __builtin_amdgcn_exp2f(fmaf(st[s][8 * c + i], c2, -m_use));
          lsum += e[i];
        }
        pf[s][c].u.x = pack_bf16x2(e[0], e[1]);
        pf[s][c].u.y = pack_bf16x2(e[2], e[3]);
        pf[s][c].u.z = pack_bf16x2(e[4], e[5]);
        pf[s][c].u.w = pack_bf16x2(e[6], e[7]);
      }
    l += lsum;
    // ---- O^T = O^T + V^T P^T -----------------------------------------------------
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const uint16_t* vrow = Vt + (dt * 32 + ql) * VT_STRIDE + 8 * g;
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          Frag8 a;
          a.u = *(const uint4*)(vrow + 32 * s + 16 * c);
          ot[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a.v, pf[s][c].v, ot[dt], 0, 0, 0);
        }
    }
  };

  if constexpr (EXTRAS) {
    // tile i of the walk: the kept first keys' tiles, then the window's (beyond the last: the
    // window's go on, whose loads are harmless reads of the last key)
    auto first_key = [&](int i) { return i < n_sink_tiles ? SINK + i * KT : kt0 + (i - n_sink_tiles) * KT; };
    const int n_all = n_sink_tiles + (k_hi - kt0 + KT - 1) / KT;
    fetch(first_key(group), 0);
    if constexpr (SETS == 2) fetch(first_key(group + groups), SECOND);
    for (int i = 0; i < n_all; i += 2 * groups) {
      const int mine = i + group;
      one_tile(first_key(mine), first_key(mine + SETS * groups), 0, std::false_type{});
      if (i + groups >= n_all) break;  // uniform over the block
      one_tile(first_key(mine + groups), first_key(mine + (1 + SETS) * groups), SECOND, std::false_type{});
    }
  } else {
    const int step = groups * KT;  // keys that the groups take at a time
    int kt = kt0;                  // the first group's
    const int ahead = group * KT;
    fetch(kt + ahead, 0);
    if constexpr (SETS == 2) fetch(kt + ahead + step, SECOND);
    if (p.window <= 0) {
      for (; kt + 2 * step - 1 <= pos0; kt += 2 * step) {
        one_tile(kt + ahead, kt + ahead + SETS * step, 0, std::true_type{});
        one_tile(kt + ahead + step, kt + ahead + (1 + SETS) * step, SECOND, std::true_type{});
      }
    }
    for (; kt < k_hi; kt += 2 * step) {  // the tiles around the diagonal, or all of them under a window
      one_tile(kt + ahead, kt + ahead + SETS * step, 0, std::false_type{});
      if (kt + step >= k_hi) break;  // uniform
      one_tile(kt + ahead + step, kt + ahead + (1 + SETS) * step, SECOND, std::false_type{});
    }
  }

  // the two halves of the wave hold different keys of the same query
  l += __shfl_xor(l, 32, WAVE);
  if (GROUPS == 2 && groups == 2) {
    // the second group's sums go to the first through LDS, each thread's to the thread of the same queries
    static_assert(GROUPS == 1 || (DT * 16 + 2) * 256 * sizeof(float) <= sizeof(tiles_lds), "the sums fit where the tiles were");
    float* const sums = (float*)tiles_lds + tid;
    __syncthreads();  // no tile is read any more
    if (group == 1) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) sums[(dt * 16 + r) * 256] = ot[dt][r];
      sums[DT * 16 * 256] = m, sums[(DT * 16 + 1) * 256] = l;
    }
    __syncthreads();
    if (group == 1) return;
    const float m1 = sums[DT * 16 * 256], both = fmaxf(m, m1), to = both == -INFINITY ? 0.f : both;
    const float w0 = exp2f(m - to), w1 = exp2f(m1 - to);  // (a group without a key of this query: zero)
    l = l * w0 + sums[(DT * 16 + 1) * 256] * w1;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) ot[dt][r] = ot[dt][r] * w0 + sums[(dt * 16 + r) * 256] * w1;
    m = both;
  }
  if (q_live) {
    // (m is in units of log 2)
    if (p.sinks) l += exp2f(fmaf(p.sinks[h], 1.4426950408889634f, -m));
    const float inv = head_gate_of(p, row0 + qi, h) / l;
    uint16_t* orow = p.out + (size_t)(row0 + qi) * p.ldo + h * HD;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        // accumulators 4j .. 4j+3: head columns dt*32 + 8j + 4g + (0..3)
        float w[4] = {inv, inv, inv, inv};
        if (EXTRAS && p.gate) {
          const uint2 gv = *(const uint2*)(p.gate + (size_t)(row0 + qi) * p.ldg + h * HD + dt * 32 + 8 * j + 4 * g);
          const float gf[4] = {__uint_as_float(gv.x << 16), __uint_as_float(gv.x & 0xffff0000u),
                               __uint_as_float(gv.y << 16), __uint_as_float(gv.y & 0xffff0000u)};
#pragma unroll
          for (int c = 0; c < 4; ++c) w[c] = inv / (1.0f + expf(-gf[c]));
        }
        uint2 o;
        o.x = pack_bf16x2(ot[dt][4 * j] * w[0], ot[dt][4 * j + 1] * w[1]);
        o.y = pack_bf16x2(ot[dt][4 * j + 2] * w[2], ot[dt][4 * j + 3] * w[3]);
        *(uint2*)(orow + dt * 32 + 8 * j + 4 * g) = o;
      }
  }
}

// ---------------------------------------------------------------------------
// Heads of 64 without optional terms of a score, in pages of a power of two of sixteen keys or more: one page then holds
// the sixteen keys of a tile that a wave copies.
//
// The same blocks, walks and arithmetic as above.  What differs is how a tile comes to its products, so that the vector
// unit has little to do but the softmax:
//  * Keys and values go from the pages to LDS by copies (lds_copy.h), two copies of a kilobyte a wave and tile for
//    each, into rings of three tiles, keys asked for three tiles ahead and values two; a page's place is three scalar instructions out of a table in LDS.
//    Before, a tile went through registers: a dozen integer instructions an address and 24 to transpose the values.
//  * Values are transposed by the LDS read (ds_read_b64_tr_b16: four keys of a column a lane).  A lane's eight scores of a
//    chunk are keys 4 g .. + 3 and 8 + 4 g .. + 3 of it, and two such reads bring the values of just these.
//  * A row's pieces of 16 bytes lie permuted (piece ^ (row / 2 % 8) of keys, piece ^ 4 (row / 2 % 2) of values), so that the
//    sixteen rows of a read of keys, and the four rows x 64 bytes of a read of values, meet all banks: no conflict is counted.
//  * The next tile's scores are begun while this one's probabilities are made, in the registers that are free by then, so
//    that a wave needs fewer registers than the 168 of three waves a SIMD and three blocks share a CU.  (With the scores in two sets of
//    registers, a whole tile ahead, 232: two blocks, 8 % more for 8,000 tokens.)
// 25 heads of 64 in pages of sixteen, us, the kernel above and this one: 8,000 tokens 317 and 259 (0.79 PFLOP/s of the causal half), under
// a window of 1,000 110 and 87; 2 x 1,024 23.7 and 20.2; 512 on 4,000 earlier keys 58.9 and 49.9; 512 12.8 and 10.9; 333 10.4 and
// 9.4; eight portions of 128 on 300 earlier keys under a window of 77 12.0 and 11.1; 40 on 500 under one of 100 8.4 and 8.4; 17 4.7 and
// 4.9 (its outputs' way through LDS, below).  What bounds it: vector instructions, 74 % of the CUs' cycles beside 41 % for the products
// (8,000 tokens at 1.88 GHz); at few blocks the way to the first tile and the walk's steps of some 1 us.

typedef short i16x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4_t* lds_i16x4_p;
union FragHalves {
  i16x4_t h[2];
  bf16x8_t v;
};
// Four keys of one column a lane: lane l of each sixteen names four columns (8 bytes) of key l / 4 and gets column l of
// all four keys.
__device__ __forceinline__ i16x4_t read_transposed(uint32_t at) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4_p)(uintptr_t)at);
}
__device__ __forceinline__ bf16x8_t read_piece(uint32_t at) {
  return *(const __attribute__((address_space(3))) bf16x8_t*)(uintptr_t)at;
}
// The larger of a value and the one of the lane 32 away (the maximum as an instruction: fmaxf first makes its operands
// canonical, which these are).  The swap exchanges halves of two registers and says nothing of one register with itself, so
// the second operand is made a value of its own, which the compiler cannot put where the first one lies.
__device__ __forceinline__ float max_of_halves(float v) {
  uint32_t mine = __float_as_uint(v), copy = mine;
  asm("" : "+v"(copy));
  const auto r = __builtin_amdgcn_permlane32_swap(mine, copy, false, false);
  float larger;
  asm("v_max_f32 %0, %1, %2" : "=v"(larger) : "v"(r[0]), "v"(r[1]));
  return larger;
}

// Head h of tile `tile`'s queries.  ring: LDS for the tiles, ring_bytes(GROUPS) of it; page_at: [max_blocks], byte offsets of this
// head's part of the request's pages, from the first tile's on.
constexpr int ring_bytes(int groups) { return groups * 2 * 3 * KT * 128; }
template <int HD, int GROUPS>
__device__ __forceinline__ void attend_tile(const PrefillArgs& p, int h, int tile, char* ring, size_t* page_at) {
  constexpr int DC = HD / 16, DT = HD / 32;
  constexpr int ROW = HD * 2, WAVE_KEYS = KT / 4, COPIES = WAVE_KEYS * ROW / 1024;  // bytes a key; keys and copies a wave and tile
  constexpr int SLOTS = 3, TILE = KT * ROW, GROUP_LDS = 2 * SLOTS * TILE;
  static_assert(HD == 64, "the permutations of a row's pieces are those of rows of 128 bytes");
  static_assert(GROUPS * GROUP_LDS == ring_bytes(GROUPS), "the kernels' LDS");

  const int group = GROUPS > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
  const int tid = threadIdx.x & 255, lane = tid & 63;  // (within the group)
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row0 = p.tiles[2 * tile];
  const int nq = p.tiles[2 * tile + 1];
  const int kv_head = h / (p.n_heads / p.n_kv_heads);
  const int pos0 = __builtin_amdgcn_readfirstlane(p.positions[row0]), request = __builtin_amdgcn_readfirstlane(p.token_req[row0]);
  asm volatile("" ::"s"(pos0), "s"(request));  // (one wait for the two: left alone, the second load stands behind the first's use)
  const int* table = p.block_table + (size_t)request * p.max_blocks;

  const int ql = lane & 31, g = lane >> 5;
  const int qi = wave * 32 + ql;  // this lane's query within the tile
  const bool q_live = qi < nq;
  const int qpos = pos0 + qi;
  const int q_lo = p.window > 0 ? max(0, qpos - p.window + 1) : 0;

  // (a lane without a query takes the last one's: nothing of it is stored)
  Frag8 qf[DC];
  {
    const uint16_t* qrow = p.q + (size_t)(row0 + min(qi, nq - 1)) * p.ldq + h * HD + 8 * g;
#pragma unroll
    for (int dc = 0; dc < DC; ++dc) qf[dc].u = *(const uint4*)(qrow + dc * 16);
  }

  const int k_hi = pos0 + nq;  // one past the last key any query of the tile sees
  const int k_lo = p.window > 0 ? max(0, pos0 - p.window + 1) : 0;
  const int kt0 = (k_lo / KT) * KT;
  const int n_tiles = (k_hi - kt0 + KT - 1) / KT;
  // (in a short walk the second group's waves end here: barriers count the waves that are left)
  const int groups = GROUPS > 1 && n_tiles >= TWO_GROUPS_FROM<HD> ? GROUPS : 1;
  if (GROUPS > 1 && group >= groups) return;
  const int n_steps = (n_tiles + groups - 1) / groups;
  // keys this wave's queries can see end here (a wave without queries: none)
  const int wave_hi = wave * 32 < nq ? min(k_hi, pos0 + wave * 32 + 32) : 0;
  const int wave_q0 = pos0 + wave * 32;  // position of the wave's first query
  const float c2 = p.scale * 1.4426950408889634f;  // scores to units of log 2

  const int shift = p.page_shift, row_mask = p.page_size - 1;
  const int pg0 = kt0 >> shift, n_pg = ((k_hi - 1) >> shift) - pg0 + 1, first_page = k_lo >> shift;
  for (int i = threadIdx.x; i < n_pg; i += 256 * groups)
    page_at[i] = ((size_t)(uint32_t)table[max(pg0 + i, first_page)] * p.page_stride + (size_t)(kv_head << shift) * HD) * 2;
  __syncthreads();

  // (the queries are waited for here, ahead of the copies: the compiler, which does not count those, would wait for all)
#pragma unroll
  for (int dc = 0; dc < DC; ++dc) asm volatile("" : "+v"(qf[dc].v));

  // Copies: this wave brings keys 16 wave .. + 15 of each tile, which lie in one page.  Of keys beyond the last, and of the
  // first tile's keys before the first that any query sees, nothing is read, and zeros come: such keys enter the products with a
  // weight of zero, and what lies there (another request's keys, infinities) must not make NaN of it.
  const uint32_t ring_at = lds_address(ring) + group * GROUP_LDS;
  const uint32_t copy_at = __builtin_amdgcn_readfirstlane(ring_at + wave * COPIES * 1024);
  const int row8 = lane >> 3;
  const uint32_t k_from0 = row8 * ROW + (((lane & 7) ^ (row8 >> 1)) * 16), k_from1 = row8 * ROW + (((lane & 7) ^ (4 + (row8 >> 1))) * 16);
  const uint32_t v_from = row8 * ROW + (((lane & 7) ^ (4 * ((row8 >> 1) & 1))) * 16);
  auto first_key = [&](int t) __attribute__((always_inline)) { return kt0 + (t * groups + group) * KT; };
  auto page_entry = [&](int t) __attribute__((always_inline)) {
    return page_at[min(((first_key(t) + wave * WAVE_KEYS) >> shift) - pg0, n_pg - 1)];
  };
  // where this wave's keys of tile t lie in the pages, and how many bytes of them there are
  struct Source {
    uint32_t lo, hi;
    int bytes;
  };
  auto source = [&](int t, size_t entry) __attribute__((always_inline)) {
    const int key = first_key(t) + wave * WAVE_KEYS;
    const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)entry), hi = __builtin_amdgcn_readfirstlane((uint32_t)(entry >> 32));
    const size_t at = (((size_t)hi << 32) | lo) + (uint32_t)((key & row_mask) * ROW);
    int keys;  // (as scalar instructions: the compiler takes the vector unit's median)
    asm("s_max_i32 %0, %1, 0\n\ts_min_i32 %0, %0, %2" : "=&s"(keys) : "s"(k_hi - key), "n"(WAVE_KEYS) : "scc");
    return Source{(uint32_t)at, (uint32_t)(at >> 32), keys * ROW};
  };
  // (what a copy's descriptor is made of is the same in all lanes; the compiler loses sight of that)
  auto copy = [&](const uint16_t* pages, const Source& s, uint32_t from0, uint32_t from1, uint32_t to) __attribute__((always_inline)) {
    const size_t at = (size_t)pages + (((size_t)s.hi << 32) | s.lo);
    const i32x4_t buffer = {__builtin_amdgcn_readfirstlane((int)(uint32_t)at), __builtin_amdgcn_readfirstlane((int)((at >> 32) & 0xffffu)),
                            __builtin_amdgcn_readfirstlane(s.bytes), BUFFER_WORD3};
    copy_pair_to_lds(buffer, from0, from1, __builtin_amdgcn_readfirstlane(to));
  };
  auto copy_k = [&](const Source& s, int slot) __attribute__((always_inline)) { copy(p.k_pages, s, k_from0, k_from1, copy_at + slot * TILE); };
  auto copy_v = [&](const Source& s, int slot) __attribute__((always_inline)) { copy(p.v_pages, s, v_from, v_from, copy_at + (SLOTS + slot) * TILE); };

  float m = -INFINITY, l = 0.f;
  f32x16_t ot[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) ot[dt][r] = 0.f;

  // where this lane reads: keys (rows of S^T's first operand) and, transposed, values
  uint32_t k_read[DC], v_read[DT];
#pragma unroll
  for (int dc = 0; dc < DC; ++dc) k_read[dc] = ring_at + ql * ROW + (((2 * dc + g) ^ ((ql >> 1) & 7)) * 16);
  const int vrow = 4 * g + ((lane & 15) >> 2);
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
    v_read[dt] = ring_at + SLOTS * TILE + vrow * ROW +
                 (((4 * dt + 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) ^ (4 * ((vrow >> 1) & 1))) * 16) + (lane & 1) * 8;

  // (an address whose origin the compiler does not see: what is added to it goes into the reads' offsets)
  auto opaque = [](uint32_t at) __attribute__((always_inline)) {
    asm("" : "+v"(at));
    return at;
  };
  auto read_k = [&](bf16x8_t (&kf)[2], uint32_t at) __attribute__((always_inline)) {  // of both subtiles
#pragma unroll
    for (int s = 0; s < 2; ++s) kf[s] = read_piece(at + s * 32 * ROW);
  };
  auto read_v = [&](bf16x8_t (&vf)[DT], int c, const uint32_t (&at)[DT]) __attribute__((always_inline)) {  // of keys 16 c .. + 15
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      FragHalves f;
#pragma unroll
      for (int e = 0; e < 2; ++e) f.h[e] = read_transposed(at[dt] + (16 * c + 8 * e) * ROW);
      vf[dt] = f.v;
    }
  };
  const f32x16_t NO_SUMS = {};
  auto scores = [&](f32x16_t (&sn)[2], int slot) __attribute__((always_inline)) {
    bf16x8_t kf[DC][2];
#pragma unroll
    for (int dc = 0; dc < DC; ++dc) read_k(kf[dc], opaque(k_read[dc] + slot * TILE));
#pragma unroll
    for (int dc = 0; dc < DC; ++dc)
#pragma unroll
      for (int s = 0; s < 2; ++s) sn[s] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[dc][s], qf[dc].v, dc == 0 ? NO_SUMS : sn[s], 0, 0, 0);
  };
  auto rescale = [&](float tmax) __attribute__((always_inline)) {
    if (__any(tmax > m)) {
      const float m_new = fmaxf(m, tmax);
      const float alpha = __builtin_amdgcn_exp2f(m - (m_new == -INFINITY ? 0.f : m_new));  // (a row with no key yet: zero)
      l *= alpha;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) ot[dt][r] *= alpha;
      m = m_new;
    }
  };

  // One step: the softmax and the output's products of tile t out of its scores `st`, and the scores of tile t + 1 to `sn`.
  auto whole = [&](int kt) __attribute__((always_inline)) { return kt + KT - 1 <= wave_q0 && (p.window <= 0 || kt >= wave_q0 + 31 - p.window + 1); };
  // A tile that every query of the wave sees whole, with another one behind it.  Eight pieces of four scores' probabilities;
  // the products go beside them as their operands are there: the first subtile's registers take the next tile's scores
  // when its probabilities are made, the second's at the end.
  auto steady_step = [&](f32x16_t (&st)[2], int kslot, int vslot) __attribute__((always_inline)) {
    bf16x8_t kf[DC][2], vf[4][DT];
    float tmax = -INFINITY;
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int r = 0; r < 16; r += 2) tmax = fmaxf(fmaxf(st[s][r], st[s][r + 1]), tmax);
    uint32_t v_at[DT], k_at[DC];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) v_at[dt] = opaque(v_read[dt] + vslot * TILE);
#pragma unroll
    for (int dc = 0; dc < DC; ++dc) k_at[dc] = opaque(k_read[dc] + kslot * TILE);
    read_v(vf[0], 0, v_at);
    rescale(max_of_halves(tmax * c2));  // (c2 > 0: the largest score stays the largest)
    const float m_use = m == -INFINITY ? 0.f : m;
    __builtin_amdgcn_sched_barrier(0);
    Frag8 pf[4];
    float part[4];
    auto output = [&](int c) __attribute__((always_inline)) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) ot[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[c][dt], pf[c].v, ot[dt], 0, 0, 0);
    };
    auto score = [&](int s, int dc) __attribute__((always_inline)) {
      st[s] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[dc][s], qf[dc].v, dc == 0 ? NO_SUMS : st[s], 0, 0, 0);
    };
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float e[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        e[i] = __builtin_amdgcn_exp2f(fmaf(st[j >> 2][4 * (j & 3) + i], c2, -m_use));
        part[i] = j == 0 ? e[i] : part[i] + e[i];
      }
      if (j & 1)
        pf[j >> 1].u.z = pack_bf16x2(e[0], e[1]), pf[j >> 1].u.w = pack_bf16x2(e[2], e[3]);
      else
        pf[j >> 1].u.x = pack_bf16x2(e[0], e[1]), pf[j >> 1].u.y = pack_bf16x2(e[2], e[3]);
      // (what is multiplied is read from LDS two pieces earlier)
      if (j == 1) read_v(vf[1], 1, v_at);
      if (j >= 2 && j < 6) kf[j - 2][0] = read_piece(k_at[j - 2]);
      if (j == 4) read_v(vf[2], 2, v_at);
      if (j == 6) read_v(vf[3], 3, v_at);
      if (j == 2) output(0);
      if (j == 4) output(1);
      if (j >= 4) score(0, j - 4);
      if (j == 6) output(2);
      if (j >= 6) kf[j - 6][1] = read_piece(k_at[j - 6] + 32 * ROW);
      __builtin_amdgcn_sched_barrier(0);
    }
    kf[2][1] = read_piece(k_at[2] + 32 * ROW);
    kf[3][1] = read_piece(k_at[3] + 32 * ROW);
    output(3);
#pragma unroll
    for (int dc = 0; dc < DC; ++dc) score(1, dc);
    l += (part[0] + part[1]) + (part[2] + part[3]);
  };
  // Any tile; the next one's scores take the place of its own at the end.
  auto step = [&](f32x16_t (&st)[2], int t, int kslot, int vslot) __attribute__((always_inline)) {
    const int kt = first_key(t);
    const bool now = kt < wave_hi, next = first_key(t + 1) < wave_hi;
    if (now) {
      float tmax = -INFINITY;
      if (!whole(kt)) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = kt + 32 * s + 8 * (r >> 2) + 4 * g + (r & 3);
            st[s][r] = q_live && key <= qpos && key >= q_lo ? st[s][r] : -INFINITY;
          }
      }
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int r = 0; r < 16; r += 2) tmax = fmaxf(fmaxf(st[s][r], st[s][r + 1]), tmax);
      rescale(max_of_halves(tmax * c2));
      const float m_use = m == -INFINITY ? 0.f : m;
      Frag8 pf[4];
      float part[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) part[i] = 0.f;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        float e[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          e[i] = __builtin_amdgcn_exp2f(fmaf(st[c >> 1][8 * (c & 1) + i], c2, -m_use));
          part[i & 3] += e[i];
        }
        pf[c].u = make_uint4(pack_bf16x2(e[0], e[1]), pack_bf16x2(e[2], e[3]), pack_bf16x2(e[4], e[5]), pack_bf16x2(e[6], e[7]));
      }
      l += (part[0] + part[1]) + (part[2] + part[3]);
      uint32_t v_at[DT];
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) v_at[dt] = opaque(v_read[dt] + vslot * TILE);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        bf16x8_t vf[DT];
        read_v(vf, c, v_at);
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) ot[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[dt], pf[c].v, ot[dt], 0, 0, 0);
      }
    }
    if (next) scores(st, kslot);
  };

  // What is on its way when step t begins: K(t + 2), V(t + 1) and all before.  A step asks for V(t + 2) and K(t + 3),
  // into the slots of K(t) and V(t - 1), which every wave has read when the step's barrier is passed.
  static_assert(COPIES == 2, "a pair of copies a tile");
  Source ahead;  // of tile t + 2
  // (only the first tile holds keys before k_lo: rows `unseen` and less of this wave's sixteen)
  const int unseen = k_lo - first_key(0) - wave * WAVE_KEYS;
  constexpr uint32_t NOTHING = COPY_NOTHING - 1024;  // (the second copy adds its kilobyte)
  auto seen = [&](uint32_t from, int row) __attribute__((always_inline)) { return row < unseen ? NOTHING : from; };
  ahead = source(0, page_entry(0));
  copy(p.k_pages, ahead, seen(k_from0, row8), seen(k_from1, 8 + row8), copy_at);
  copy(p.v_pages, ahead, seen(v_from, row8), seen(v_from, 8 + row8), copy_at + SLOTS * TILE);
#pragma unroll
  for (int t = 1; t < 3; ++t) {
    ahead = source(t, page_entry(t));
    copy_k(ahead, t);
    if (t < 2) copy_v(ahead, t);
  }
  size_t entry = page_entry(3);  // of tile t + 3, read from LDS a step ahead
  f32x16_t sa[2];
  copies_arrived<4 * COPIES>();  // K(0): behind it V(0), K(1), V(1), K(2)
  ring_barrier();
  if (first_key(0) < wave_hi) scores(sa, 0);
  int slot = 0;  // of K(t) and V(t)
  auto turn = [&](f32x16_t (&st)[2], int t, auto steady) __attribute__((always_inline)) {
    copies_arrived<2 * COPIES>();  // K(t + 1) and V(t): behind them K(t + 2) and V(t + 1)
    ring_barrier();
    const int before = slot == 0 ? SLOTS - 1 : slot - 1, after = slot == SLOTS - 1 ? 0 : slot + 1;
    copy_v(ahead, before);
    ahead = source(t + 3, entry);
    copy_k(ahead, slot);
    entry = page_entry(t + 4);
    if constexpr (decltype(steady)::value)
      steady_step(st, after, slot);
    else
      step(st, t, after, slot);
    slot = after;
  };
  // The steps from `from` up to `to` are of tiles that every query of the wave sees whole, with another one behind.  (The waves of a block go through theirs each on its own; what they share is a barrier a step.)
  const int key0 = first_key(0), step_keys = groups * KT;
  const int seen_from = p.window > 0 ? max(wave_q0 + 32 - p.window - key0, 0) : 0;
  const int from = (seen_from + step_keys - 1) / step_keys;
  const int seen_to = min(wave_q0 + 1 - KT, wave_hi - 1 - step_keys) - key0;  // the last one's first key
  const int to = seen_to < 0 ? 0 : seen_to / step_keys + 1;
  for (int t = 0; t < n_steps; ++t) {
    if (t >= from)
      for (; t < to; ++t) turn(sa, t, std::true_type{});
    turn(sa, t, std::false_type{});
  }
  copies_arrived<0>();  // (what was asked for beyond the last tile)

  // the two halves of the wave hold different keys of the same query
  l += __shfl_xor(l, 32, WAVE);
  if (GROUPS == 2 && groups == 2) {
    // the second group's sums go to the first through LDS, each thread's to the thread of the same queries
    static_assert(GROUPS == 1 || (DT * 16 + 2) * 256 * sizeof(float) <= GROUPS * GROUP_LDS, "the sums fit where the tiles were");
    float* const sums = (float*)ring + tid;
    __syncthreads();  // no tile is read any more
    if (group == 1) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) sums[(dt * 16 + r) * 256] = ot[dt][r];
      sums[DT * 16 * 256] = m, sums[(DT * 16 + 1) * 256] = l;
    }
    __syncthreads();
    if (group == 1) return;
    const float m1 = sums[DT * 16 * 256], both = fmaxf(m, m1), to = both == -INFINITY ? 0.f : both;
    const float w0 = exp2f(m - to), w1 = exp2f(m1 - to);  // (a group without a key of this query: zero)
    l = l * w0 + sums[(DT * 16 + 1) * 256] * w1;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int r = 0; r < 16; ++r) ot[dt][r] = ot[dt][r] * w0 + sums[(dt * 16 + r) * 256] * w1;
    m = both;
  }
  // (m is in units of log 2)
  if (p.sinks) l += exp2f(fmaf(p.sinks[h], 1.4426950408889634f, -m));
  const float inv = head_gate_of(p, row0 + min(qi, nq - 1), h) / l;
  // The outputs leave through LDS, as whole rows of 128 bytes that go through to memory: stored as they lie here, pieces of
  // 8 bytes of 32 rows, they had to stay in the L2s and were written back at the kernel's end (2 x 1,024 tokens of 25 heads
  // 22.2 -> 21.1 us, 512 11.5 -> 10.6, 8,000 271 -> 264, under a window of 1,000 97 -> 86.5; 17 4.8 -> 5.0: that sitting's figures).
  constexpr int OUT_ROW = ROW + 16;  // bytes from row to row in LDS: sixteen rows' pieces on different banks
  static_assert(4 * 32 * OUT_ROW <= GROUP_LDS, "the outputs fit where the tiles were");
  if (GROUPS == 1) __syncthreads();  // no tile is read any more (of two groups: where the second one's tiles were, which end above)
  char* const rows_at = ring + (GROUPS - 1) * GROUP_LDS + wave * 32 * OUT_ROW;
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // accumulators 4j .. 4j+3: head columns dt*32 + 8j + 4g + (0..3)
      uint2 o;
      o.x = pack_bf16x2(ot[dt][4 * j] * inv, ot[dt][4 * j + 1] * inv);
      o.y = pack_bf16x2(ot[dt][4 * j + 2] * inv, ot[dt][4 * j + 3] * inv);
      *(uint2*)(rows_at + ql * OUT_ROW + (dt * 32 + 8 * j + 4 * g) * 2) = o;
    }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();  // (a wave's rows are its own, and its LDS accesses keep their order)
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int row = s * 8 + row8, q = wave * 32 + row;
    if (q >= nq) continue;
    const u32x4_t o = *(const u32x4_t*)(rows_at + row * OUT_ROW + (lane & 7) * 16);
    uint16_t* const to = p.out + (size_t)(row0 + q) * p.ldo + h * HD + (lane & 7) * 8;
    if (p.out_by_16) {
      store_through(to, o);
    } else {
      *(uint2*)to = make_uint2(o.x, o.y);
      *(uint2*)(to + 4) = make_uint2(o.z, o.w);
    }
  }
}

template <int HD, int GROUPS>
__global__ __launch_bounds__(256 * GROUPS) __attribute__((amdgpu_waves_per_eu(GROUPS == 1 ? 3 : 2, GROUPS == 1 ? 3 : 2)))
void attn_prefill_ring_kernel(PrefillArgs p) {
  __shared__ __attribute__((aligned(1024))) char ring[ring_bytes(GROUPS)];
  extern __shared__ size_t page_at[];
  attend_tile<HD, GROUPS>(p, blockIdx.x, blockIdx.y, ring, page_at);
}

// A prompt's portion and the rows that decode beside it in one launch: first the tiles' blocks, a few long ones bound by their
// instructions, then the rows', many that wait for memory, both in blocks of four waves, three a CU.  One after the other, as
// two launches, the second waited for the last block of the first.  25 heads, us, two launches and one: 24 rows at 200 to
// 900 keys beside 512 tokens 32.1 and 22.5 (the rows alone 20.7), beside 16 24.6 and 20.4, beside 1,000 38.1 and 26.4; 48 rows at 16 to 900
// beside 512 41.7 and 31.8; 11 rows at 30 to 60 beside 1,000 22.8 and 19.6.  What bounds it: the rows' keys, then the tiles' walks.
template <int HD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) void attn_mixed_kernel(PrefillArgs p, DecodeArgs rows, int n_tiles) {
  __shared__ __attribute__((aligned(1024))) char ring[ring_bytes(1)];
  extern __shared__ size_t page_at[];
  const int lin = blockIdx.x, item = lin / p.n_heads, h = lin - item * p.n_heads;  // (a row's heads are neighbours, as in the decode kernel)
  if (item < n_tiles) {
    attend_tile<HD, 1>(p, h, item, ring, page_at);
  } else {
    attend_row<uint16_t, HD / 8, true, false, 4, false>(rows, __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), 4, item - n_tiles, h, 0, nullptr);
  }
}

DEFINE_LAST_ERROR(mlxlm_last_error)

// The longest table that attn_mixed takes (the walks themselves are not known where a step is recorded).  Its tiles go by one group of
// waves a block, and where few short rows stand beside a walk of some 2,000 keys that costs what the launch saves or a little
// more; us, two launches and one, 512 tokens on 1,500 earlier keys: beside 11 rows at 30 to 60 keys, 25 heads, 32.5 and 32.3, 4 heads
// 30.0 and 31.0; beside 8 at 200 to 1,000 38.4 and 32.6, 33.5 and 30.9; beside 24 at 200 to 900 47.3 and 35.6, 34.5 and 31.1; at 200 to 2,000
// 64.8 and 44.8, 25 heads; 1,000 on 1,024 beside 24 at 30 to 60 34.7 and 32.2, 29.4 and 30.1; 16 on 2,000 beside 11 at 30 to 60 29.0 and
// 27.1, 27.6 and 26.3.  Longer walks are not measured in one launch.
#define MIXED_MOST_KEYS 2048
// And the longest row where the decode kernel would give rows eight waves or parts, which are sooner done alone: one row of 700
// keys beside 16 / 512 / 1,000 tokens 13.1, 19.9, 26.1 (eight waves) and 11.0, 12.2, 19.1 in one launch; four at 200 to 900 14.6,
// 21.5, 27.7 and 13.5, 14.3, 19.2; eight at 200 to 1,000 16.3, 22.9, 29.3 and 15.7, 16.2, 19.6: level beside the fewest tokens
// (of 2 heads, whose rows go in parts alone, 12.5 and 13.2 beside 16).
#define MIXED_MOST_ROW_KEYS 1024

// tiles: n_tiles pairs (first flat row, number of rows 1..128); the rows of a
// tile are consecutive tokens of one request at consecutive positions.
// bfloat16 only, head_dim 32, 64, 128 or 256.
static int prefill_launch(void* out, const void* q, int ldq, int ldo, const void* k_pages,
                          const void* v_pages, size_t page_stride, const int* block_table,
                          int max_blocks, const int* token_req, const int* positions,
                          const int* tiles, int n_tiles, int n_heads, int n_kv_heads,
                          int head_dim, int page_size, int window, float scale,
                          const float* head_scale, const float* slopes, const void* gate, int ldg,
                          int keep_first, const AttnTerms* shape, hipStream_t stream, const int* rows = nullptr, int n_rows = 0) {
  if (n_tiles <= 0) return 0;
  if (shape && (shape->softcap < 0.f || (shape->dist_bias && shape->n_dist <= 0)))
    FAIL("attn_prefill: softcap %g, a distance table of %d entries a head", (double)shape->softcap, shape->n_dist);
  if (keep_first < 0) FAIL("attn_prefill: keep_first %d must not be negative", keep_first);
  if (gate && (ldg < n_heads * head_dim || ldg % 4 != 0 || ((uintptr_t)gate & 7)))
    FAIL("attn_prefill: the gate's rows (stride %d) must be 8-byte aligned and as wide as the output's", ldg);
  if (head_dim != 32 && head_dim != 64 && head_dim != 128 && head_dim != 256)
    FAIL("attn_prefill: head_dim %d is not 32, 64, 128 or 256 (attn_tile takes the others)", head_dim);
  if (n_heads <= 0 || n_kv_heads <= 0 || n_heads % n_kv_heads != 0)
    FAIL("attn_prefill: %d query heads cannot be grouped over %d key heads", n_heads, n_kv_heads);
  if (page_size <= 0) FAIL("attn_prefill: page_size %d must be positive", page_size);
  if (!out || !q || !k_pages || !v_pages || !block_table || !token_req || !positions || !tiles)
    FAIL("attn_prefill: null pointer");
  if (ldq % 8 != 0 || ((uintptr_t)q & 15)) FAIL("attn_prefill: query rows must be 16-byte aligned");
  if (ldo % 4 != 0 || ((uintptr_t)out & 7)) FAIL("attn_prefill: output rows must be 8-byte aligned");
  if (page_stride % 8 != 0 || (((uintptr_t)k_pages | (uintptr_t)v_pages) & 15))
    FAIL("attn_prefill: pages must be 16-byte aligned");
  if (window < 0) FAIL("attn_prefill: window %d must not be negative", window);
  if (page_stride >= ((size_t)1 << 32)) FAIL("attn_prefill: a page of %zu elements is too large", page_stride);
  PrefillArgs p;
  p.out = (uint16_t*)out, p.q = (const uint16_t*)q;
  p.out_by_16 = ldo % 8 == 0 && !((uintptr_t)out & 15);
  p.k_pages = (const uint16_t*)k_pages, p.v_pages = (const uint16_t*)v_pages;
  p.block_table = block_table, p.token_req = token_req, p.positions = positions, p.tiles = tiles;
  p.page_stride = page_stride, p.ldq = ldq, p.ldo = ldo, p.max_blocks = max_blocks;
  p.page_shift = -1;
  for (int sh = 0; sh < 31; ++sh)
    if ((1 << sh) == page_size) p.page_shift = sh;
  p.n_heads = n_heads, p.n_kv_heads = n_kv_heads, p.page_size = page_size, p.window = window;
  p.scale = scale;
  p.head_scale = head_scale, p.slopes = slopes, p.gate = (const uint16_t*)gate, p.ldg = ldg;
  p.keep_first = window > 0 ? keep_first : 0;
  p.softcap = shape ? shape->softcap : 0.f, p.dist_bias = shape ? shape->dist_bias : nullptr;
  p.n_dist = shape ? shape->n_dist : 0;
  p.sinks = shape ? shape->sinks : nullptr, p.head_gate = shape ? shape->head_gate : nullptr;
  p.ldhg = shape ? shape->ldhg : 0;
  if (p.head_gate && p.ldhg < n_heads) FAIL("attn_prefill: the heads' gate has rows of %d columns", p.ldhg);
  const bool shaped = p.softcap > 0.f || p.dist_bias;
  const bool extras = head_scale || slopes || gate || p.keep_first > 0 || shaped;
  if (n_tiles > 65535) FAIL("attn_prefill: %d tiles in a launch, at most 65535", n_tiles);
  // a request's page numbers lie in LDS beside the tiles
  if (max_blocks > 7168)
    FAIL("attn_prefill: block tables of %d pages a request do not fit beside the tiles (at most 7168)", max_blocks);
  // (the kept first keys' pages lie before the window's; a page can be in both runs)
  const size_t lds = (size_t)(max_blocks + (extras ? 2 : 0)) * sizeof(int);
  const bool pow2 = p.page_shift >= 0;
  // (pages of one to eight keys, of which a copy of sixteen would take several, keep the general kernel and its shifts: by
  // divisions, and so without two groups, 25 heads in pages of eight took 82.7 us for 512 on 4,000 earlier keys, 57.9 with, 8,000 361 / 328)
  const bool ring = head_dim == 64 && !extras && p.page_shift >= 4;
  // Two groups a block where the blocks are no more than the CUs, so that a block's walk is the kernel's time: 1,024 tokens
  // of 25 heads of 64 (200 blocks) 19.1 us beside 21.3, 512 on 4,000 earlier keys 57 / 72, of 16 heads of 32 43 / 58.  With
  // more blocks than CUs they are in each other's way (2 x 1,024 tokens of 25 heads, 400 blocks: 25.5 / 23.1; 4 x 512:
  // 20.7 / 15.2).  The kernel for heads of 64 without terms, one row of figures each: 1,024 16.9 / 18.4, 512 on 4,000 49 / 59.4;
  // 2 x 1,024 23.2 / 20.8, 4 x 512 18.4 / 13.5.  Heads of 128 and more take the registers of a whole SIMD a wave.
  const bool two = head_dim <= 64 && pow2 && max_blocks <= 4096 && (long)n_heads * n_tiles <= n_compute_units();
  const dim3 grid(n_heads, n_tiles), block(two ? 512 : 256);
#define LAUNCH_AS(HD, POW2, GROUPS)                                                                                      \
  do {                                                                                                                  \
    if (shaped)                                                                                                         \
      hipLaunchKernelGGL((attn_prefill_kernel<HD, POW2, true, true, GROUPS>), grid, block, lds, stream, p);             \
    else if (extras)                                                                                                    \
      hipLaunchKernelGGL((attn_prefill_kernel<HD, POW2, true, false, GROUPS>), grid, block, lds, stream, p);            \
    else                                                                                                                \
      hipLaunchKernelGGL((attn_prefill_kernel<HD, POW2, false, false, GROUPS>), grid, block, lds, stream, p);           \
  } while (0)
#define LAUNCH_PREFILL(HD)              \
  do {                                  \
    if (two) {                          \
      LAUNCH_AS(HD, true, (HD <= 64 ? 2 : 1)); \
    } else if (pow2) {                  \
      LAUNCH_AS(HD, true, 1);           \
    } else {                            \
      LAUNCH_AS(HD, false, 1);          \
    }                                   \
  } while (0)
  if (rows) {  // (attn_mixed has looked at what the rows need beyond this)
    if (!ring) FAIL("attn_mixed: pages of %d keys", page_size);
    DecodeArgs d = {};
    d.out = out, d.q = q, d.k_pages = k_pages, d.v_pages = v_pages;
    d.block_table = block_table, d.token_req = token_req, d.positions = positions, d.rows = rows;
    d.page_stride = page_stride, d.ldq = ldq, d.ldo = ldo, d.max_blocks = max_blocks;
    d.n_heads = n_heads, d.n_kv_heads = n_kv_heads, d.page_size = page_size, d.window = window, d.n_splits = 1;
    d.scale = scale, d.out_head_dim = head_dim, d.table_in_lds = 1, d.page_shift = p.page_shift;
    hipLaunchKernelGGL((attn_mixed_kernel<64>), dim3((unsigned)(n_heads * (n_tiles + n_rows))), dim3(256), (size_t)max_blocks * sizeof(size_t), stream, p, d, n_tiles);
  } else if (ring) {
    const size_t table = (size_t)max_blocks * sizeof(size_t);
    if (two)
      hipLaunchKernelGGL((attn_prefill_ring_kernel<64, 2>), grid, block, table, stream, p);
    else
      hipLaunchKernelGGL((attn_prefill_ring_kernel<64, 1>), grid, block, table, stream, p);
  } else if (head_dim == 32) {
    LAUNCH_PREFILL(32);
  } else if (head_dim == 64) {
    LAUNCH_PREFILL(64);
  } else if (head_dim == 128) {
    LAUNCH_PREFILL(128);
  } else {
    LAUNCH_PREFILL(256);
  }
#undef LAUNCH_PREFILL
#undef LAUNCH_AS
  CHECK_LAUNCH("attn_prefill");
  return 0;
}

// 1 if attn_mixed takes a step's tiles and rows, of which the longest reads `row_keys`: bfloat16 heads of 64 with a key head
// each; rows that the decode kernel would give four waves a block too (more (row, head)s than CUs), or short ones.
extern "C" int attn_mixed_takes(int n_tiles, int n_rows, int n_heads, int n_kv_heads, int head_dim, int page_size, int max_blocks,
                                long row_keys) {
  return n_tiles > 0 && n_rows > 0 && n_tiles + n_rows <= 65535 && head_dim == 64 && n_heads == n_kv_heads && page_size >= 16 &&
         (page_size & (page_size - 1)) == 0 && (long)max_blocks * page_size <= MIXED_MOST_KEYS &&
         ((long)n_rows * n_heads > n_compute_units() || row_keys <= MIXED_MOST_ROW_KEYS);
}

// attn_prefill's tiles and attn_decode_rows' rows, of one step, in one launch.
extern "C" int attn_mixed(void* out, const void* q, int ldq, int ldo, const void* k_pages, const void* v_pages, size_t page_stride,
                          const int* block_table, int max_blocks, const int* token_req, const int* positions, const int* tiles, int n_tiles,
                          const int* rows, int n_rows, int n_heads, int n_kv_heads, int head_dim, int page_size, int window, float scale,
                          hipStream_t stream) {
  if (!attn_mixed_takes(n_tiles, n_rows, n_heads, n_kv_heads, head_dim, page_size, max_blocks, 0))
    FAIL("attn_mixed: %d tiles and %d rows of %d heads of %d over %d, %d pages of %d keys", n_tiles, n_rows, n_heads, head_dim, n_kv_heads,
         max_blocks, page_size);
  if (!rows || max_blocks <= 0 || ldo < n_heads * head_dim) FAIL("attn_mixed: null pointer or stride");
  return prefill_launch(out, q, ldq, ldo, k_pages, v_pages, page_stride, block_table, max_blocks, token_req, positions, tiles, n_tiles, n_heads,
                        n_kv_heads, head_dim, page_size, window, scale, nullptr, nullptr, nullptr, 0, 0, nullptr, stream, rows, n_rows);
}

// attn_prefill_biased: with the optional terms of PrefillArgs (null or 0 where one is absent).
extern "C" int attn_prefill_biased(void* out, const void* q, int ldq, int ldo, const void* k_pages,
                                   const void* v_pages, size_t page_stride, const int* block_table,
                                   int max_blocks, const int* token_req, const int* positions,
                                   const int* tiles, int n_tiles, int n_heads, int n_kv_heads,
                                   int head_dim, int page_size, int window, float scale,
                                   const float* head_scale, const float* slopes, const void* gate, int ldg,
                                   int keep_first, hipStream_t stream) {
  return prefill_launch(out, q, ldq, ldo, k_pages, v_pages, page_stride, block_table, max_blocks, token_req, positions,
                        tiles, n_tiles, n_heads, n_kv_heads, head_dim, page_size, window, scale, head_scale, slopes,
                        gate, ldg, keep_first, nullptr, stream);
}

// attn_prefill_terms: every optional term, as an AttnTerms (attention_tiles.h); null: none.
extern "C" int attn_prefill_terms(void* out, const void* q, int ldq, int ldo, const void* k_pages,
                                  const void* v_pages, size_t page_stride, const int* block_table,
                                  int max_blocks, const int* token_req, const int* positions,
                                  const int* tiles, int n_tiles, int n_heads, int n_kv_heads,
                                  int head_dim, int page_size, int window, float scale, const AttnTerms* t,
                                  hipStream_t stream) {
  return prefill_launch(out, q, ldq, ldo, k_pages, v_pages, page_stride, block_table, max_blocks, token_req, positions,
                        tiles, n_tiles, n_heads, n_kv_heads, head_dim, page_size, window, scale,
                        t ? t->head_scale : nullptr, t ? t->slopes : nullptr, t ? t->gate : nullptr, t ? t->ldg : 0,
                        t ? t->keep_first : 0, t, stream);
}

extern "C" int attn_prefill(void* out, const void* q, int ldq, int ldo, const void* k_pages,
                            const void* v_pages, size_t page_stride, const int* block_table,
                            int max_blocks, const int* token_req, const int* positions,
                            const int* tiles, int n_tiles, int n_heads, int n_kv_heads,
                            int head_dim, int page_size, int window, float scale,
                            hipStream_t stream) {
  return attn_prefill_biased(out, q, ldq, ldo, k_pages, v_pages, page_stride, block_table, max_blocks, token_req,
                             positions, tiles, n_tiles, n_heads, n_kv_heads, head_dim, page_size, window, scale,
                             nullptr, nullptr, nullptr, 0, 0, stream);
}
