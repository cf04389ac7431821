// All layers of a decode step of one or two rows as one launch: for each layer
//   q, k, v = LN(h) Wq^T + bq;  a = attention(q, cache and k, v);  h1 = h + a Wo^T + bo;
//   act = gelu(LN(h1) W1^T + b1);  h = h1 + act W2^T + b2
// (the reference runs them as operations of their own, mlx_lm/models/gpt2.py:44-80,98-108).
//
// What bounds it: so few rows cost a layer five launches of 4 to 10 us, each 1.7 us from the last
// one's end, then a trip for its rows, then its weights from memory, then the drain.  In one launch a
// hand-over between two products is one store and one load that meet in memory, 1.2 us, and the next unit's
// weights come into LDS meanwhile (keys and values, which no product of the step makes, into registers).  A wave
// that issues those copies stands still until the memory has taken them, 3 to 4 us for the 100 KB of a unit (a compute
// unit draws some 25 KB a us), and rows that it asks for come behind them: so CH_COPIERS waves of the block do nothing
// else, and the others never wait for more than their rows.  A layer of GPT-2's sizes in us, with its five launches /
// here with the computing waves copying too / with two waves to copy / with four / and the next unit looked up once (as it is):
//   width   768 at  93 keys, one row    26 / 16.3 / 16.4 / 15.7 / 15.0   (two rows, in one launch only: 18.6 / - / 17.9 / 17.8)
//   width 1,280 at 500 keys, one row    34 / 19.9 / 19.0 / 17.1 / 16.9
//   width 1,600 at 700 keys, one row    37 / 23.0 / 21.3 / 19.5 / 18.9   (two rows: 26.0 / 23.4 / 22.0 / 21.9)
// Of the 18.9 the weights' 61 MB are 9.6 at the memory's rate and the five hand-overs 6.
//
// Hand-over.  What one product hands to the next lies in words of eight bytes, 4 of payload (a float32
// of the stream, or two bfloat16) and 4 of tag; a tag belongs to one product of one step.  A word is
// stored and loaded whole, past the L2s, and a reader asks for its words again until all carry the tag
// that it waits for: the data are their own flag.  (With flags beside the data, a hand-over is the
// store's way to memory, the flag's, the poll's and the rows' own: 3.6 us, as much as a launch.  Counters
// instead of flags take 16 ns for each of some 200 additions on top.)  A word costs twice its payload and
// every block reads all rows, which is why this is for one or two rows: at 8 rows the rows of a product would
// be as many bytes as its weights.
//
// No block relies on another one running.  A unit (8 to 32 features of a product, or a row's head and part
// of the keys) belongs to a block by its number.  A wave that has waited `patience` for its words gives up: its block then
// counts the blocks that run (each says so in a word of its own) and takes its share of all units among those, from the first
// phase that lacks one; what is missing even so is done by whoever waits for it.  A unit done twice stores the
// same words twice.  A block that falls behind others on the way (its unit done by them meanwhile, and a later product's
// words in the places that it reads) sees that by their tags, and where it had read its rows already, its late words change
// nothing: a word is stored by an atomic maximum, whose high half is the tag, so what a place holds only gets later.  (With
// plain stores a late word could put back an older product's, which nobody then missed where its own product's
// successor was complete: the residual's old value would have been waited for without end.)  So a single resident block
// would finish the launch, whatever holds the rest of the GPU.  A step of XL at 700 keys with 0 / 64 / 128 / 224 of 256 compute
// units held by another stream's kernel for longer than the step (us): 1,005 / 2,149 / 2,098 / 6,168; where units kept their first
// owners 1,004 / 16,494 / 16,877 / until they were free; each layer's own launches 1,851 / 2,174 / 2,323 / 5,149.  GPT-2 small at 93
// keys pays for the first wait: 253 / 491 / 567 / 1,095 against 349 / 340 / 370 / 609.  (Blocks of twelve waves of
// 168 registers leave no room beside them: two engines' steps on two streams follow each other, a pair of XL steps 1,999
// against 2,266; beside an XL step of 8 rows the step of one row takes 989 instead of 2,384, and the pair 3,094 instead of 2,722.)
#include <atomic>

#include "decode_chain.h"
#include "lds_copy.h"

#define CH_WAVES 8         // waves that compute products
#define CH_COPIERS 4       // waves that copy the next unit's weights meanwhile
#define CH_ALL_WAVES (CH_WAVES + CH_COPIERS)  // (attention is everybody's)
#define CH_LN_BLOCKS 4     // k-blocks (64) a wave of a normed product holds: K <= 2,048
#define CH_PAIRS 7         // pairs of k-blocks a wave of the other products holds: K <= 7,168
#define CH_TILES 2         // tiles of 16 features a unit of a normed product has at most
#define CH_HELD 8          // pairs of fragments of weights a wave holds
#define CH_LN_MOST (CH_LN_BLOCKS * CH_WAVES * 64)
#define CH_COPY_MOST (CH_PAIRS * CH_WAVES * 128)
#define CH_HEAD CHAIN_HEAD_DIM
#define CH_TAGS_A_STEP 0x10000u  // more than a step has products
#define CH_KEY_TILES ((CHAIN_MOST_KEYS + CH_ALL_WAVES * 8 - 1) / (CH_ALL_WAVES * 8))  // loads of 8 keys a wave holds

#define CH_LDS_MOST (160 * 1024)
#define CH_DEVICES 64  // whose grants of LDS are remembered (others ask at each launch)
// Ticks of 10 ns.  200 us: some five times the longest wait of any size (a head's, for a layer of width
// 2,048, 38 us); 100 and 60 were 0.1 ms better for held compute units and worse beside short kernels, whose places come free
// (XL beside large products, nine steps of ten within 1.4 ms, then 1.75 and 1.9).  Dealt anew, a wait is a phase's, and 30 us
// are enough: with 10 a step of 2.3 ms took 2.8 (blocks that wait for a head did others' units).
#define CH_PATIENCE 20000
#define CH_PATIENCE_ANEW 3000u
#define CH_UNITS_MOST 4096u  // a phase has fewer: 3 x 7,168 features of q, k and v, 8 a unit

enum { CH_QKV = 0, CH_ATTN, CH_OUT, CH_FC, CH_PROJ, CH_KINDS };

struct ChainSize {
  int N, K, features, units;
};
typedef unsigned long long word_t;  // payload in the low half, tag in the high
struct ChainArgs {
  const ChainLayer* layers;
  int n_layers;
  ChainSize size[CH_KINDS];
  int product_blocks, attention_blocks;  // attention's are the later ones
  word_t* present;  // a word a block: tag_base's once it runs
  const uint32_t* tag_base;
  uint32_t patience;   // ticks of 10 ns
  float eps1, eps2, scale;
  const float* h;      // rows in (the embedding) and rows out, [R][ldh]
  float* h_out;
  int ldh;
  // words, a row after the other
  word_t* qkv;   // pairs
  word_t* att;   // pairs
  word_t* h1;
  word_t* act;   // pairs
  word_t* h2;
  int n_heads, n_kv_heads, q_width, kv_width, page_size, max_blocks;
  size_t page_stride;
  const int* block_table;
  const int* token_req;
  const int* positions;
};

typedef u32x4_t ChFrag;  // eight bfloat16 of a matrix instruction's operand
__device__ __forceinline__ f32x4_t mfma(ChFrag a, ChFrag b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

__device__ __forceinline__ word_t word_load(const word_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// (a maximum: a place that holds a later product's word keeps it)
__device__ __forceinline__ void word_store(word_t* p, uint32_t payload, uint32_t tag) {
  (void)__hip_atomic_fetch_max(p, ((word_t)tag << 32) | payload, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void word_store(word_t* p, float payload, uint32_t tag) { word_store(p, __float_as_uint(payload), tag); }
__device__ __forceinline__ uint32_t tag_of(word_t w) { return (uint32_t)(w >> 32); }
__device__ __forceinline__ float f32_of(word_t w) { return __uint_as_float((uint32_t)w); }

// How a wait ended: the words are there, nobody stored them for `patience`, or a later product's are in their places.
enum { CH_THERE = 0, CH_MISSING = 1, CH_LATE = 2 };

// Load words with `load(i)` until all `n` (<= MOST, the wave's own) of all lanes carry `tag`.  (Two rounds of loads on
// their way at a time, half a trip apart, were slower: 18.6 us a layer of width 768 instead of 16.3.)
template <int MOST, typename F>
__device__ __forceinline__ int words_wait(word_t (&w)[MOST], int n, uint32_t tag, uint32_t patience, F load) {
  uint64_t since = 0;
  for (;;) {
    // (a word that this wave does not have counts as there: nothing is then carried from one round to the next in registers)
#pragma unroll
    for (int i = 0; i < MOST; ++i) {
      w[i] = (word_t)tag << 32;
      if (i < n) w[i] = load(i);
    }
    bool there = true, late = false;
#pragma unroll
    for (int i = 0; i < MOST; ++i) {
      there = there && tag_of(w[i]) == tag;
      late = late || tag_of(w[i]) > tag;
    }
    if (__all(there)) return CH_THERE;
    if (__any(late)) return CH_LATE;
    const uint64_t now = wall_clock64();
    if (since == 0) since = now;
    if (now - since >= patience) return CH_MISSING;
    __builtin_amdgcn_s_sleep(1);
  }
}

__device__ __forceinline__ int ceil_of(int a, int b) { return (a + b - 1) / b; }

// What a product's unit reads that no unit of the step makes (weights, bias, the norm's scale and shift) comes
// into LDS by copies of 1 KB, dealt to the copying waves.  Fragment h of tile t and k-block c of a normed
// product lies at ((t * k-blocks + c) * 2 + h) KB, half h of pair c of a plain one at (c * 2 + h) KB; scale and shift lie as
// the computing waves read them, each its own k-blocks'.
// (the table of layers is read by scalar loads: nothing writes it during a launch)
typedef const __attribute__((address_space(4))) ChainLayer* layer_ptr;
__device__ __forceinline__ layer_ptr layer_of(const ChainArgs& p, int layer) { return (layer_ptr)(uintptr_t)(p.layers + layer); }
struct ChainUnit {
  int kind, which, n0, n_end, kblocks, pairs, n_blocks, n_pairs;  // (the last two: this wave's)
  bool normed;
  layer_ptr ly;
};
__device__ __forceinline__ ChainUnit unit_of(const ChainArgs& p, int ph, int unit, int wave) {
  ChainUnit x;
  x.kind = ph % CH_KINDS, x.which = x.kind == CH_QKV ? 0 : x.kind - 1;
  x.normed = x.kind == CH_QKV || x.kind == CH_FC;
  const ChainSize& z = p.size[x.kind];
  x.n0 = unit * z.features, x.n_end = min(x.n0 + z.features, z.N);
  x.kblocks = z.K >> 6, x.pairs = (x.kblocks + 1) >> 1;
  x.n_blocks = (x.kblocks - wave + CH_WAVES - 1) / CH_WAVES;
  x.n_pairs = (x.pairs - wave + CH_WAVES - 1) / CH_WAVES;
  x.ly = layer_of(p, ph / CH_KINDS);
  return x;
}
__device__ __forceinline__ void copy_unit(const ChainArgs& p, const ChainUnit& x, uint32_t lds, uint32_t lds_small, int lane, int copier) {
  const int g = lane >> 4;
  const ChainSize& z = p.size[x.kind];
  const i32x4_t from = copy_buffer(x.ly->W[x.which], (size_t)((z.N + 15) / 16) * x.kblocks * 2048);
  if (copier == 0 && x.ly->bias[x.which])
    copy16_to_lds(copy_buffer(x.ly->bias[x.which], (size_t)z.N * 4), lane < 8 && x.n0 + lane * 4 < z.N ? (x.n0 + lane * 4) * 4 : COPY_NOTHING, 0,
                  lds_small + CH_WAVES * 2048);
  if (x.normed) {
    const i32x4_t gamma = copy_buffer(x.ly->gamma[x.kind == CH_FC], (size_t)z.K * 4), beta = copy_buffer(x.ly->beta[x.kind == CH_FC], (size_t)z.K * 4);
    for (int v = copier; v < CH_WAVES; v += CH_COPIERS) {
      const int k = (v + CH_WAVES * (lane >> 4)) * 64 + (lane & 15) * 4;
      const uint32_t at = k < z.K ? k * 4 : COPY_NOTHING;
      copy16_to_lds(gamma, at, 0, lds_small + v * 2048);
      copy16_to_lds(beta, at, 0, lds_small + v * 2048 + 1024);
    }
    for (int c = copier; c < x.kblocks; c += CH_COPIERS)
#pragma unroll
      for (int t = 0; t < CH_TILES; ++t)
        if (x.n0 + t * 16 < x.n_end) {
          const int n = min(x.n0 + t * 16 + (lane & 15), x.n_end - 1);
          const uint32_t at = (uint32_t)(n >> 4) * x.kblocks * 2048 + (g * 16 + (n & 15)) * 16;
          copy16_to_lds(from, at, c * 2048, lds + (t * x.kblocks + c) * 2048);
          copy16_to_lds(from, at, c * 2048 + 1024, lds + (t * x.kblocks + c) * 2048 + 1024);
        }
  } else {
    // 8 features; a matrix instruction takes them at two k-blocks at once (rows 0 to 7 of the
    // weights and of the rows' columns the first, 8 to 15 the second; the products of one's
    // weights with the other's rows are not used)
    const int n = x.n0 + (lane & 7);
    const uint32_t at = (uint32_t)(n >> 4) * x.kblocks * 2048 + (g * 16 + (n & 15)) * 16, second = (lane >> 3) & 1;
    for (int pair = copier; pair < x.pairs; pair += CH_COPIERS) {
      const uint32_t at2 = !second ? at : 2 * pair + 1 < x.kblocks ? at + 2048 : COPY_NOTHING;  // (no second k-block: zeros)
      copy16_to_lds(from, at2, pair * 4096, lds + pair * 2048);
      copy16_to_lds(from, at2, pair * 4096 + 1024, lds + pair * 2048 + 1024);
    }
  }
}

// A barrier of the computing waves alone (the copying ones are held up by their copies): `arrived` counts, `target`
// is a wave's own.
__device__ __forceinline__ void meet(uint32_t* arrived, uint32_t& target, int lane) {
  target += CH_WAVES;
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  if (lane == 0) atomicAdd(arrived, 1u);
  while ((int)(*(volatile uint32_t*)arrived - target) < 0) {
  }
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// Sum (largest) over the lanes that hold the same eighth (lane % 8) of different keys.
__device__ __forceinline__ float keys_sum(float v) {
  v += dpp_move<0x128>(v);  // row_ror:8
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}
__device__ __forceinline__ float keys_max(float v) {
  v = fmaxf(v, dpp_move<0x128>(v));
  v = fmaxf(v, __shfl_xor(v, 16, 64));
  return fmaxf(v, __shfl_xor(v, 32, 64));
}

template <int R>
struct ChainShared {
  __attribute__((aligned(16))) uint16_t xs[R][CH_COPY_MOST + 8];
  float red[CH_TILES][CH_WAVES][2 * R * 16];
  __attribute__((aligned(16))) float small[CH_WAVES * 2 + 1][256];  // the norm's scale and shift, a wave's own share; the bias
  __attribute__((aligned(16))) float4 stat[R][CH_WAVES];
  __attribute__((aligned(16))) float part[CH_ALL_WAVES][CH_HEAD];
  float part_m[16], part_l[16];
  int how[CH_ALL_WAVES];
  uint32_t missing;
  // what the block does next, for all waves: phase (-1: no more) and unit, whether its weights are in LDS, and the unit after it
  struct {
    int ph, unit, held, then_ph, then_unit, anew;
  } plan;
  // Dealt anew: this block's place among those that run and their number, a missing unit that it does in its own's stead, and
  // the unit whose weights are in LDS or on their way
  struct {
    int start, stride, help_i, help_u, held_ph, held_unit;
  } anew;
  uint32_t arrived;
};

// One unit of attention: a row's head.  Old keys lie in the pages and are asked for before the step's query
// is there; the step's own key and value come in words, and go to their page from here.
template <int R>
__device__ __forceinline__ int chain_attention(const ChainArgs& p, ChainShared<R>& sh, int layer, int u, uint32_t tag, uint32_t patience,
                                               int lane, int wave) {
  const int h = u % p.n_heads, m = u / p.n_heads, kvh = h / (p.n_heads / p.n_kv_heads);
  const layer_ptr ly = layer_of(p, layer);
  const int pos = p.positions[m];
  const int* table = p.block_table + (size_t)p.token_req[m] * p.max_blocks;
  const int tiles = ceil_of(pos, 8), e = lane & 7;
  // a lane holds 8 of a key's 64 elements, a load 8 keys; wave w takes tiles w, w + 12, ...
  const auto place = [&](int key) {
    return (size_t)table[key / p.page_size] * p.page_stride + ((size_t)kvh * p.page_size + key % p.page_size) * CH_HEAD + e * 8;
  };
  ChFrag k[CH_KEY_TILES], v[CH_KEY_TILES];
  float sc[CH_KEY_TILES], mine = -INFINITY, top = -INFINITY;
#pragma unroll
  for (int t = 0; t < CH_KEY_TILES; ++t) k[t] = v[t] = (ChFrag)(0u), sc[t] = -INFINITY;
#pragma unroll
  for (int t = 0; t < CH_KEY_TILES; ++t) {
    if (t * CH_ALL_WAVES + wave >= tiles) break;
    const size_t at = place(min((t * CH_ALL_WAVES + wave) * 8 + (lane >> 3), pos - 1));
    k[t] = *(const ChFrag*)((const uint16_t*)ly->k_pages + at), v[t] = *(const ChFrag*)((const uint16_t*)ly->v_pages + at);
  }
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);

  const word_t* row = p.qkv + (size_t)m * (p.size[CH_QKV].N >> 1);
  word_t in[12];
  const bool own = wave == CH_ALL_WAVES - 1;  // the wave that takes the step's own key
  const int how = words_wait(in, own ? 12 : 4, tag - 1, patience, [&](int i) {
    const int first = i < 4 ? h * CH_HEAD : p.q_width + (i >= 8 ? p.kv_width : 0) + kvh * CH_HEAD;
    return word_load(row + ((first + e * 8) >> 1) + (i & 3));
  });
  float q[8];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    q[2 * j] = __uint_as_float((uint32_t)in[j] << 16) * p.scale;
    q[2 * j + 1] = __uint_as_float((uint32_t)in[j] & 0xffff0000u) * p.scale;
  }
  const auto score = [&](uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
    const uint32_t kk[4] = {a, b, c, d};
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      s = __builtin_fmaf(q[2 * j], __uint_as_float(kk[j] << 16), s);
      s = __builtin_fmaf(q[2 * j + 1], __uint_as_float(kk[j] & 0xffff0000u), s);
    }
    return group_sum<8>(s);
  };
#pragma unroll
  for (int t = 0; t < CH_KEY_TILES; ++t) {
    if (t * CH_ALL_WAVES + wave >= tiles) break;
    const float s = score(k[t][0], k[t][1], k[t][2], k[t][3]);
    sc[t] = (t * CH_ALL_WAVES + wave) * 8 + (lane >> 3) < pos ? s : -INFINITY;
    top = fmaxf(top, sc[t]);
  }
  if (own) {
    const float s = score((uint32_t)in[4], (uint32_t)in[5], (uint32_t)in[6], (uint32_t)in[7]);
    if (lane < 8) mine = s;
    top = fmaxf(top, mine);
  }
  top = keys_max(top);
  float o[8], l = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = 0.f;
  const float base = top == -INFINITY ? 0.f : top;  // (a wave without keys)
#pragma unroll
  for (int t = 0; t < CH_KEY_TILES; ++t) {
    if (t * CH_ALL_WAVES + wave >= tiles) break;
    const float w = __builtin_amdgcn_exp2f(sc[t] - base);
    l += w;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      o[2 * j] = __builtin_fmaf(w, __uint_as_float(v[t][j] << 16), o[2 * j]);
      o[2 * j + 1] = __builtin_fmaf(w, __uint_as_float(v[t][j] & 0xffff0000u), o[2 * j + 1]);
    }
  }
  if (own && lane < 8) {
    const float w = __builtin_amdgcn_exp2f(mine - base);
    l += w;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      o[2 * j] = __builtin_fmaf(w, __uint_as_float((uint32_t)in[8 + j] << 16), o[2 * j]);
      o[2 * j + 1] = __builtin_fmaf(w, __uint_as_float((uint32_t)in[8 + j] & 0xffff0000u), o[2 * j + 1]);
    }
  }
  l = keys_sum(l);
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = keys_sum(o[j]);
  if (lane < 8) {
    *(float4*)(&sh.part[wave][e * 8]) = make_float4(o[0], o[1], o[2], o[3]);
    *(float4*)(&sh.part[wave][e * 8 + 4]) = make_float4(o[4], o[5], o[6], o[7]);
  }
  if (lane == 0) sh.part_m[wave] = top, sh.part_l[wave] = l, sh.how[wave] = how;
  __syncthreads();
  int worst = 0;
#pragma unroll
  for (int w = 0; w < CH_ALL_WAVES; ++w) worst |= sh.how[w];
  worst = __builtin_amdgcn_readfirstlane(worst);
  if (wave == 0 && worst == CH_THERE) {
    const int w16 = lane & 15;
    const float m_w = w16 < CH_ALL_WAVES ? sh.part_m[w16] : -INFINITY, best = group_max<16>(m_w);
    const float f = m_w == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_w - best);
    const float inv = 1.0f / group_sum<16>(f == 0.f ? 0.f : f * sh.part_l[w16]);
    float out = 0.f;
#pragma unroll
    for (int w = 0; w < CH_ALL_WAVES; ++w) out = __builtin_fmaf(lane_value(f, w), sh.part[w][lane], out);
    out *= inv;
    const float next = dpp_move<DPP_QUAD_SWAP1>(out);
    if ((lane & 1) == 0) word_store(p.att + (((size_t)m * p.q_width + h * CH_HEAD + lane) >> 1), pack_bf16x2(out, next), tag);
  }
  if (own && lane < 8 && worst == CH_THERE) {
    const size_t at = place(pos);
    *(ChFrag*)((uint16_t*)ly->k_pages + at) = (ChFrag){(uint32_t)in[4], (uint32_t)in[5], (uint32_t)in[6], (uint32_t)in[7]};
    *(ChFrag*)((uint16_t*)ly->v_pages + at) = (ChFrag){(uint32_t)in[8], (uint32_t)in[9], (uint32_t)in[10], (uint32_t)in[11]};
  }
  return worst;
}

extern __shared__ __attribute__((aligned(16))) char held_weights[];

// A unit of a product.  Computing waves return how their wait for rows ended; copying ones leave with the weights of the unit
// after it on their way.
template <int R>
__device__ __forceinline__ int chain_product(const ChainArgs& p, ChainShared<R>& sh, int ph, int unit, bool in_lds, int then_ph, int then_unit,
                                             uint32_t tag, uint32_t patience, uint32_t& target, int lane, int wave) {
  const uint32_t lds = lds_address(held_weights), lds_small = lds_address(sh.small);
  const int kind = ph % CH_KINDS, layer = ph / CH_KINDS;
  const bool copies = wave >= CH_WAVES;
  if (!in_lds) {
    if (copies) {
      copy_unit(p, unit_of(p, ph, unit, wave), lds, lds_small, lane, wave - CH_WAVES);
      copies_arrived<0>();
    }
    __syncthreads();
  }
  if (copies) {
    __syncthreads();  // (the computing waves have read what lies in LDS)
    if (then_ph >= 0) copy_unit(p, unit_of(p, then_ph, then_unit, wave), lds, lds_small, lane, wave - CH_WAVES);
    return CH_THERE;
  }
  const ChainUnit at_hand = unit_of(p, ph, unit, wave);
  const ChainSize& z = p.size[kind];
  const bool normed = at_hand.normed, first = ph == 0, last = ph == p.n_layers * CH_KINDS - 1;
  const int g = lane >> 4, kblocks = at_hand.kblocks, pairs = at_hand.pairs, n_blocks = at_hand.n_blocks, n_pairs = at_hand.n_pairs;
  const int n0 = at_hand.n0, n_end = at_hand.n_end;
  const bool odd = kblocks & 1;  // the last pair has no second k-block: its lanes repeat the first, and count as zeros
  const bool short_pair = odd && n_pairs > 0 && wave + CH_WAVES * (n_pairs - 1) == pairs - 1;

  // ---- what the copying waves brought ---------------------------------------------------------
  // wave 0 writes the outputs: one feature a lane into the stream, else two neighbours a lane
  const int o_m = normed ? lane >> 4 : lane >> 3;
  const int o_f = normed ? (lane & 15) * 2 : lane & 7;
  const bool mine = wave == 0 && o_m < R && n0 + o_f < n_end;
  float2 bias = make_float2(0.f, 0.f);
  float old = 0.f;
  if (wave == 0 && at_hand.ly->bias[at_hand.which]) bias.x = sh.small[CH_WAVES * 2][o_f], bias.y = sh.small[CH_WAVES * 2][o_f + 1];
  float gm[CH_LN_BLOCKS], bt[CH_LN_BLOCKS];
#pragma unroll
  for (int b = 0; b < CH_LN_BLOCKS; ++b) gm[b] = sh.small[wave * 2][b * 64 + lane], bt[b] = sh.small[wave * 2 + 1][b * 64 + lane];
  ChFrag w[CH_HELD][2];
#pragma unroll
  for (int b = 0; b < CH_HELD; ++b) w[b][0] = w[b][1] = (ChFrag)(0u);
  if (normed) {
#pragma unroll
    for (int t = 0; t < CH_TILES; ++t)
      if (n0 + t * 16 < n_end)
#pragma unroll
        for (int b = 0; b < CH_LN_BLOCKS; ++b)
          if (b < n_blocks) {
            const char* at = held_weights + (t * kblocks + wave + CH_WAVES * b) * 2048 + lane * 16;
            w[t * CH_LN_BLOCKS + b][0] = *(const ChFrag*)at, w[t * CH_LN_BLOCKS + b][1] = *(const ChFrag*)(at + 1024);
          }
    asm volatile("; weights of a normed product" ::: "memory");  // (the branches' ends differ: merged, w would be indexed by a variable)
  } else {
#pragma unroll
    for (int b = 0; b < CH_PAIRS; ++b)
      if (b < n_pairs) {
        const char* at = held_weights + (wave + CH_WAVES * b) * 2048 + lane * 16;
        w[b][0] = *(const ChFrag*)at, w[b][1] = *(const ChFrag*)(at + 1024);
      }
    asm volatile("; weights of a plain product" ::: "memory");
  }
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();  // the copying waves go on with the next unit's

  // ---- the rows, and the products ----------------------------------------------------------
  int how = CH_THERE;
  f32x4_t acc[CH_TILES];
#pragma unroll
  for (int t = 0; t < CH_TILES; ++t) acc[t] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
  if (normed) {
    float x[R][CH_LN_BLOCKS];
    if (first) {
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int b = 0; b < CH_LN_BLOCKS; ++b)
          x[r][b] = b < n_blocks ? p.h[(size_t)r * p.ldh + (wave + CH_WAVES * b) * 64 + lane] : 0.f;
    } else {
      word_t in[R * CH_LN_BLOCKS];
      const word_t* from = (kind == CH_QKV ? p.h2 : p.h1) + wave * 64;
      how |= words_wait(in, n_blocks * R, tag - 1, patience, [&](int j) {  // (word j: row j % R of block j / R)
        return word_load(from + ((j % R) * z.K + (j / R) * (CH_WAVES * 64)) + (uint32_t)lane);
      });
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int b = 0; b < CH_LN_BLOCKS; ++b) x[r][b] = b < n_blocks ? f32_of(in[b * R + r]) : 0.f;
    }
    // The wave's own mean and squares around it, then all waves' joined in one exchange (squares around
    // a wave's mean are as exact as around the row's): n (mean_w - mean)^2 comes on top.
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float s = 0.f;
#pragma unroll
      for (int b = 0; b < CH_LN_BLOCKS; ++b) s += x[r][b];
      s = wave_sum(s);
      const float wmean = s * (n_blocks == 4 ? 0x1p-8f : n_blocks == 3 ? 1.f / 192.f : n_blocks == 2 ? 0x1p-7f : 0x1p-6f);
      float qq = 0.f;
#pragma unroll
      for (int b = 0; b < CH_LN_BLOCKS; ++b) {
        const float d = x[r][b] - wmean;
        qq += b < n_blocks ? d * d : 0.f;
      }
      qq = wave_sum(qq);
      if (lane == 0) sh.stat[r][wave] = make_float4(s, wmean, qq, (float)(n_blocks * 64));
    }
    meet(&sh.arrived, target, lane);
    const float inv_k = 1.0f / (float)z.K;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float4 st = sh.stat[r][lane & 7];
      const float mean = group_sum<8>(st.x) * inv_k;
      const float d = st.y - mean;
      const float var = group_sum<8>(st.z + st.w * d * d) * inv_k + (kind == CH_QKV ? p.eps1 : p.eps2);
      float rstd = __builtin_amdgcn_rsqf(var);
      rstd = rstd * (1.5f - 0.5f * var * rstd * rstd);  // (the instruction is an ulp off, one step is not)
#pragma unroll
      for (int b = 0; b < CH_LN_BLOCKS; ++b)
        if (b < n_blocks)
          sh.xs[r][(wave + CH_WAVES * b) * 64 + lane] = f32_to_bf16_bits((x[r][b] - mean) * rstd * gm[b] + bt[b]);
    }
    // (a wave reads back only what it wrote itself)
    const uint16_t* xr = sh.xs[min(lane & 15, R - 1)] + g * 16;
#pragma unroll
    for (int b = 0; b < CH_LN_BLOCKS; ++b) {
      const int c = wave + CH_WAVES * b;
      if (b < n_blocks) {
        const ChFrag a0 = *(const ChFrag*)(xr + c * 64), a1 = *(const ChFrag*)(xr + c * 64 + 8);
#pragma unroll
        for (int t = 0; t < CH_TILES; ++t) {
          acc[t] = mfma(w[t * CH_LN_BLOCKS + b][0], a0, acc[t]);
          acc[t] = mfma(w[t * CH_LN_BLOCKS + b][1], a1, acc[t]);
        }
      }
    }
  } else {
    // word 0: the stream's old value, wave 0's alone (complete long before the rows, and waited for all the same: its
    // tag is made this one); then word j: row (j - 1) % R of pair (j - 1) / R
    const int whole = short_pair && lane >= 32 ? n_pairs - 1 : n_pairs;  // pairs that this lane's words exist of
    word_t in[R * CH_PAIRS + 1];
    const word_t* from = (kind == CH_OUT ? p.att : p.act) + wave * 64;
    const bool from_rows = kind == CH_OUT && layer == 0;
    const size_t old_at = (size_t)min(o_m, R - 1) * z.N + min(n0 + o_f, z.N - 1);
    if (wave == 0 && from_rows) old = p.h[(size_t)min(o_m, R - 1) * p.ldh + min(n0 + o_f, z.N - 1)];
    how |= words_wait(in, whole * R + 1, tag - 1, patience, [&](int j) {
      if (j > 0) return word_load(from + ((j - 1) % R * (z.K >> 1) + (j - 1) / R * (CH_WAVES * 64)) + (uint32_t)lane);
      if (wave != 0 || from_rows) return (word_t)(tag - 1) << 32;
      return kind == CH_OUT ? word_load(p.h2 + old_at) + ((word_t)2 << 32) : word_load(p.h1 + old_at) + ((word_t)1 << 32);
    });
    if (wave == 0 && !from_rows) old = f32_of(in[0]);
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int b = 0; b < CH_PAIRS; ++b)
        if (b < whole) *(uint32_t*)(sh.xs[r] + (wave + CH_WAVES * b) * 128 + lane * 2) = (uint32_t)in[b * R + r + 1];
    const int r = min(lane & 7, R - 1), second = (lane >> 3) & 1;
#pragma unroll
    for (int b = 0; b < CH_PAIRS; ++b) {
      const int pair = wave + CH_WAVES * b;
      if (pair < pairs) {
        const bool repeats = odd && pair == pairs - 1 && second;
        const uint16_t* from = sh.xs[r] + pair * 128 + (repeats ? 0 : second * 64) + g * 16;
        ChFrag x0 = *(const ChFrag*)from, x1 = *(const ChFrag*)(from + 8);
        if (repeats) x0 = x1 = (ChFrag)(0u);
        acc[0] = mfma(w[b][0], x0, acc[0]);
        acc[0] = mfma(w[b][1], x1, acc[0]);
      }
    }
  }

  // ---- the waves' tiles are added by wave 0 in a fixed order; element: row t / 16, feature t % 16 ----
  // (only rows that are there are kept: column m, and for the pairs' second k-blocks column m + 8)
#pragma unroll
  for (int t = 0; t < CH_TILES; ++t)
    if (t == 0 || n0 + t * 16 < n_end)
      if ((lane & 7) < R)
#pragma unroll
        for (int r = 0; r < 4; ++r) sh.red[t][wave][((lane >> 3 & 1) * R + (lane & 7)) * 16 + 4 * g + r] = acc[t][r];
  if (lane == 0) sh.how[wave] = how;
  meet(&sh.arrived, target, lane);
  int worst = 0;
#pragma unroll
  for (int v = 0; v < CH_WAVES; ++v) worst |= sh.how[v];
  worst = __builtin_amdgcn_readfirstlane(worst);
  if (mine && worst == CH_THERE) {
    if (!normed) {
      float v = 0.f;
#pragma unroll
      for (int k = 0; k < CH_WAVES; ++k) v += sh.red[0][k][o_m * 16 + o_f] + sh.red[0][k][(o_m + R) * 16 + o_f + 8];
      v = old + (v + bias.x);
      if (last)
        p.h_out[(size_t)o_m * p.ldh + n0 + o_f] = v;
      else
        word_store((kind == CH_OUT ? p.h1 : p.h2) + (size_t)o_m * z.N + n0 + o_f, v, tag);
    } else {
      const int tile = o_f >> 4, f = o_f & 15, n = n0 + o_f;
      float v0 = 0.f, v1 = 0.f;
#pragma unroll
      for (int k = 0; k < CH_WAVES; ++k) v0 += sh.red[tile][k][o_m * 16 + f], v1 += sh.red[tile][k][o_m * 16 + f + 1];
      v0 += bias.x, v1 += bias.y;
      if (kind == CH_FC) v0 = gelu_tanh_fast(v0), v1 = gelu_tanh_fast(v1);
      word_store((kind == CH_FC ? p.act : p.qkv) + (((size_t)o_m * z.N + n) >> 1), pack_bf16x2(v0, v1), tag);
    }
  }
  return worst;
}

// A plan for a block that waited for `patience`, or came so late that its unit's places held a later product's words: every
// phase's units, attention's too, are dealt among the blocks that run, counted again a layer, as others may come.  (Wave 0's.  Its
// state lies in LDS: in registers it would cost the ordinary step 2 % at two rows.)
template <int R>
__device__ __forceinline__ void plan_anew(const ChainArgs& p, ChainShared<R>& sh, uint32_t tag_base, int& i, int& u, int lane) {
  const int n_phases = p.n_layers * CH_KINDS;
  int start = __builtin_amdgcn_readfirstlane(sh.anew.start), stride = __builtin_amdgcn_readfirstlane(sh.anew.stride);
  int held_ph = __builtin_amdgcn_readfirstlane(sh.anew.held_ph), held_unit = __builtin_amdgcn_readfirstlane(sh.anew.held_unit);
  const int help_i = __builtin_amdgcn_readfirstlane(sh.anew.help_i), help_u = __builtin_amdgcn_readfirstlane(sh.anew.help_u);
  // The last phase's units stay their first owners': nobody would miss one.  (The first blocks are those with a second unit of
  // a product, so the heads go to the last.)
  const auto first_unit = [&](int at_i) {
    if (at_i == n_phases - 1) return (int)blockIdx.x < p.product_blocks ? (int)blockIdx.x : 0x7fff;
    return at_i % CH_KINDS == CH_ATTN ? stride - 1 - start : start;
  };
  const auto settle = [&](int& at_i, int& at_u) {  // to the next phase that has a unit of this block's
    while (at_i < n_phases && at_u >= p.size[at_i % CH_KINDS].units) ++at_i, at_u = first_unit(at_i);
  };
  if (start >= 0) settle(i, u);
  if (help_i < 0 && (start < 0 || (i < n_phases && i % CH_KINDS == CH_QKV && u == start))) {
    if (start < 0) {  // a phase that has begun: those ahead of the one before it are whole
      const word_t* words = lane == CH_QKV ? p.qkv : lane == CH_ATTN ? p.att : lane == CH_OUT ? p.h1 : lane == CH_FC ? p.act : p.h2;
      int front = (int)(tag_of(word_load(words)) - tag_base);
#pragma unroll
      for (int d = 1; d < 8; d *= 2) front = max(front, __shfl_xor(front, d, 64));
      i = max(__builtin_amdgcn_readfirstlane(front) - 1, 0);
    }
    int before = 0, here = 0;  // (the block's own word may still be on its way)
    for (int b = 0; b < (int)gridDim.x; b += 64) {
      const int of = b + lane;
      const uint64_t runs = __ballot(of == (int)blockIdx.x || (of < (int)gridDim.x && tag_of(word_load(p.present + min(of, (int)gridDim.x - 1))) == tag_base));
      here += __popcll(runs), before += __popcll(runs & __ballot(of < (int)blockIdx.x));
    }
    start = before, stride = here, u = first_unit(i);
    settle(i, u);
  }
  int then_i = i, then_u = u;
  if (help_i < 0) then_u += i != n_phases - 1 ? stride : p.product_blocks, settle(then_i, then_u);
  const int ph = i >= n_phases ? -1 : help_i >= 0 ? help_i : i, unit = help_i >= 0 ? help_u : u;
  const bool in_lds = ph == held_ph && unit == held_unit, copying = ph % CH_KINDS != CH_ATTN;
  if (copying) {  // the next product's weights come meanwhile (a head's unit leaves them where they are)
    held_ph = then_i, held_unit = then_u;
    while (held_ph < n_phases && held_ph % CH_KINDS == CH_ATTN) held_unit += stride, settle(held_ph, held_unit);
    if (held_ph >= n_phases) held_ph = -1;
  }
  if (lane == 0) {
    sh.plan.ph = ph, sh.plan.unit = unit, sh.plan.held = in_lds;
    sh.plan.then_ph = copying ? held_ph : -1, sh.plan.then_unit = held_unit;
    sh.anew.start = start, sh.anew.stride = stride, sh.anew.held_ph = held_ph, sh.anew.held_unit = held_unit;
  }
}

template <int R>
__global__ __launch_bounds__(CH_ALL_WAVES * 64, 3) void decode_chain_kernel(ChainArgs p) {
  __shared__ ChainShared<R> sh;
  bool held = false;  // the weights of the unit at hand are in LDS, or on their way
  bool anew = false;  // dealt anew (plan_anew)
  const int n_phases = p.n_layers * CH_KINDS;
  const uint32_t tag_base = *p.tag_base;
  const bool attends = (int)blockIdx.x >= p.product_blocks;
  // this block's next unit: `u` of phase `i` (layer i / 5, kind i % 5)
  const int start = attends ? blockIdx.x - p.product_blocks : blockIdx.x;
  const int stride = attends ? p.attention_blocks : p.product_blocks;
  int i = attends ? CH_ATTN : CH_QKV, u = start;
  const auto settle = [&] {  // to the next phase that has a unit of this block's
    while (i < n_phases && u >= p.size[i % CH_KINDS].units) u = start, i += attends ? CH_KINDS : i % CH_KINDS == CH_QKV ? 2 : 1;
  };
  settle();
  uint32_t target = 0;  // of the computing waves' own barrier
  if (threadIdx.x == 0) sh.arrived = 0, sh.plan.anew = 0, word_store(p.present + blockIdx.x, 0u, tag_base);
  for (;;) {
    // (made anew for every unit: what is computed from them would otherwise be kept in registers over the loop, 50 of them)
    int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    asm volatile("" : "+v"(lane), "+s"(wave));
    const bool copies = wave >= CH_WAVES;
    if (wave == 0 && !anew) {
      const int ph = i < n_phases ? i : -1, unit = u;
      u += stride, settle();
      const bool more = !attends && i < n_phases;
      if (lane == 0) sh.plan.ph = ph, sh.plan.unit = unit, sh.plan.held = held, sh.plan.then_ph = more ? i : -1, sh.plan.then_unit = u;
      held = more;
    } else if (wave == 0) {
      plan_anew<R>(p, sh, tag_base, i, u, lane);
    }
    if (copies) copies_arrived<0>();
    __syncthreads();
    const int ph = __builtin_amdgcn_readfirstlane(sh.plan.ph), unit = __builtin_amdgcn_readfirstlane(sh.plan.unit);
    const int then_ph = __builtin_amdgcn_readfirstlane(sh.plan.then_ph), then_unit = __builtin_amdgcn_readfirstlane(sh.plan.then_unit);
    const bool in_lds = __builtin_amdgcn_readfirstlane(sh.plan.held) != 0;
    if (ph < 0) break;
    const uint32_t patience = __builtin_amdgcn_readfirstlane(sh.plan.anew) ? min(p.patience, CH_PATIENCE_ANEW) : p.patience;
    int worst;
    if (ph % CH_KINDS == CH_ATTN) {
      worst = chain_attention<R>(p, sh, ph / CH_KINDS, unit, tag_base + ph, patience, lane, wave);
      __syncthreads();
    } else {
      worst = chain_product<R>(p, sh, ph, unit, in_lds, then_ph, then_unit, tag_base + ph, patience, target, lane, wave);
    }
    if (copies) continue;
    if (!anew) {
      if (worst == CH_THERE) continue;
      anew = true;
      if (threadIdx.x == 0) sh.anew.start = -1, sh.anew.help_i = -1, sh.anew.held_ph = -1, sh.plan.anew = 1;
      continue;
    }
    if (worst != CH_MISSING) {  // (done, or somebody else's long ago: later words lie in the places that it reads)
      if (wave == 0 && __builtin_amdgcn_readfirstlane(sh.anew.help_i) < 0)
        u += i != n_phases - 1 ? __builtin_amdgcn_readfirstlane(sh.anew.stride) : p.product_blocks;
      if (threadIdx.x == 0) sh.anew.help_i = -1;
      continue;
    }
    // Somebody's unit is missing: back to the last phase that lacks nothing, and of the one after it one missing unit, a
    // different one from block to block (the next after a block's own number was the same one for all that looked).
    if (threadIdx.x == 0) sh.anew.help_i = -1;
    for (int q = ph - 1; q >= 0; --q) {
      const int qk = q % CH_KINDS;
      const ChainSize zq = p.size[qk];
      const bool pairs_of = qk != CH_OUT && qk != CH_PROJ;
      const int per = (qk == CH_ATTN ? p.q_width : zq.N) >> (pairs_of ? 1 : 0);
      const word_t* words = qk == CH_QKV ? p.qkv : qk == CH_ATTN ? p.att : qk == CH_OUT ? p.h1 : qk == CH_FC ? p.act : p.h2;
      if (threadIdx.x == 0) sh.missing = 0xffffffffu;
      meet(&sh.arrived, target, lane);
      for (int j = threadIdx.x; j < per * R; j += CH_WAVES * 64) {
        if (tag_of(word_load(words + j)) >= tag_base + q) continue;
        const int of = qk == CH_ATTN ? (j / per) * p.n_heads + (j % per) * 2 / CH_HEAD : (j % per) * (pairs_of ? 2 : 1) / zq.features;
        atomicMin(&sh.missing, (((uint32_t)of * 0x9e3779b1u + blockIdx.x * 0x85ebca6bu) * 0xc2b2ae35u & ~(CH_UNITS_MOST - 1u)) | (uint32_t)of);
      }
      meet(&sh.arrived, target, lane);
      const uint32_t found = __builtin_amdgcn_readfirstlane(sh.missing);
      meet(&sh.arrived, target, lane);
      if (found == 0xffffffffu) break;
      if (threadIdx.x == 0) sh.anew.help_i = q, sh.anew.help_u = found & (CH_UNITS_MOST - 1);
    }
  }
}

// (a launch of its own ahead of the step's: no block may see the tag change.)  Tags only grow, as the words' maximum wants
// it: where 32 bits end, after some 18 million steps of 48 layers, the words start from zeros again.
__global__ __launch_bounds__(256) void chain_step_kernel(uint32_t* base, uint32_t by, word_t* words, int n_words) {
  const uint32_t old = *base;
  const bool again = old > 0u - 2 * CH_TAGS_A_STEP;
  __syncthreads();
  if (again)
    for (int i = threadIdx.x; i < n_words; i += 256) words[i] = 0;
  if (threadIdx.x == 0) *base = again ? by : old + by;
}

DEFINE_LAST_ERROR(mlxlm_last_error)


static bool aligned16(const void* q) { return ((uintptr_t)q & 15) == 0; }

// How a launch deals its units: `attention` blocks at the grid's end take the heads, the others the products' features,
// as few a unit as give each block one.
struct ChainDeal {
  int blocks, attention;
  ChainSize size[CH_KINDS];
  size_t lds;
};
static bool deal_of(const ChainDims* d, int rows, ChainDeal* deal) {
  const int cus = n_compute_units(), q_width = d->n_heads * CH_HEAD, kv_width = d->n_kv_heads * CH_HEAD;
  deal->blocks = cus;
  deal->attention = rows * d->n_heads < cus / 4 ? rows * d->n_heads : cus / 4;
  const int products = cus - deal->attention;
  const int n[CH_KINDS] = {q_width + 2 * kv_width, 0, d->width, d->inner, d->width};
  const int k[CH_KINDS] = {d->width, 0, q_width, d->width, d->inner};
  const size_t fixed = rows == 1 ? sizeof(ChainShared<1>) : sizeof(ChainShared<2>);
  deal->lds = 0;
  for (int i = 0; i < CH_KINDS; ++i) {
    ChainSize& z = deal->size[i];
    z.N = n[i], z.K = k[i], z.features = 8;
    if (i == CH_ATTN) {
      z.units = rows * d->n_heads;
      continue;
    }
    const int kb = z.K / 64;
    size_t held = (size_t)((kb + 1) / 2) * 2048;
    if (i == CH_QKV || i == CH_FC) {
      while (z.features < CH_TILES * 16 && (z.N + z.features - 1) / z.features > products) z.features += 8;
      held = (size_t)((z.features + 15) / 16) * kb * 2048;
      if (fixed + held > CH_LDS_MOST) z.features = 16, held = (size_t)kb * 2048;
    }
    z.units = (z.N + z.features - 1) / z.features;
    // Two rows of width 1,664 and more leave LDS for 16 features a unit only, and blocks with two units a product wait for both
    // (us a step of 12 layers at 3 / 500 / 1,000 keys, here against each layer's launches: width 1,728 of inner size 6,784 558 /
    // 563 / 570 against 474 / 513 / 532, width 2,048 of 2,048 432 / 438 / 444 against 417 / 450 / 469; width 1,600 316 / 319 /
    // 328 against 455 / 494 / 513).  One row is ahead there too (2,048 of 6,656: 450 / 454 / 460 against 502 / 529 / 563).
    if (rows > 1 && (i == CH_QKV || i == CH_FC) && z.units > products) return false;
    if (held > deal->lds) deal->lds = held;
  }
  return fixed + deal->lds <= CH_LDS_MOST;
}

extern "C" int decode_chain_takes(const ChainDims* d, int rows) {
  if (!d || rows < 1 || rows > CHAIN_MOST_ROWS || d->n_layers < 1 || d->n_layers > 4096 || n_compute_units() < 64) return 0;
  if (d->width < 64 || d->inner < 64 || d->n_heads < 1 || d->n_heads > 4096 || d->n_kv_heads < 1 || d->page_size < 1) return 0;
  if (d->width % 64 != 0 || d->inner % 64 != 0 || d->n_heads % d->n_kv_heads != 0) return 0;
  // (the output projection's K is n_heads x 64)
  if (d->width > CH_LN_MOST || d->inner > CH_COPY_MOST || d->n_heads * CH_HEAD > CH_COPY_MOST) return 0;
  ChainDeal deal;
  return deal_of(d, rows, &deal) ? 1 : 0;
}

// The launch's memory: the tag, then the words of each product in turn, then the blocks'.
static size_t words_of(const ChainDims* d, int rows, size_t (&at)[CH_KINDS + 1]) {
  const int q_width = d->n_heads * CH_HEAD, kv_width = d->n_kv_heads * CH_HEAD;
  const size_t n[CH_KINDS] = {(size_t)(q_width + 2 * kv_width) / 2, (size_t)q_width / 2, (size_t)d->width, (size_t)d->inner / 2, (size_t)d->width};
  size_t total = 32;
  for (int i = 0; i < CH_KINDS; ++i) at[i] = total, total += (n[i] * rows + 31) / 32 * 32;
  at[CH_KINDS] = total;
  return total + n_compute_units();
}
extern "C" size_t decode_chain_bytes(const ChainDims* d, int rows) {
  size_t at[CH_KINDS + 1];
  return words_of(d, rows, at) * sizeof(word_t);
}

extern "C" int decode_chain(const ChainDims* d, int rows, const void* layers, void* memory, const float* h, float* h_out, int ldh,
                            const int* block_table, int max_blocks, const int* token_req, const int* positions, int blocks,
                            unsigned patience, hipStream_t stream) {
  if (!decode_chain_takes(d, rows)) FAIL("decode_chain: sizes that this launch does not take");
  if (!layers || !memory || !h || !h_out || h == h_out || !block_table || !token_req || !positions) FAIL("decode_chain: null pointer, or h in place");
  if (!aligned16(memory) || !aligned16(layers) || ldh < d->width || max_blocks < 1 || blocks < 0) FAIL("decode_chain: alignment, row stride %d or block table", ldh);
  ChainDeal deal;
  deal_of(d, rows, &deal);
  ChainArgs a = {};
  size_t at[CH_KINDS + 1];
  const size_t n_words = words_of(d, rows, at);
  word_t* words = (word_t*)memory;
  a.layers = (const ChainLayer*)layers, a.n_layers = d->n_layers;
  for (int i = 0; i < CH_KINDS; ++i) a.size[i] = deal.size[i];
  if (blocks > 0 && blocks < deal.blocks) {  // (too few for a block of its own for attention: its units are then always missing)
    deal.blocks = blocks;
    if (deal.attention > blocks / 4) deal.attention = blocks / 4;
  }
  a.product_blocks = deal.blocks - deal.attention, a.attention_blocks = deal.attention;
  a.tag_base = (const uint32_t*)memory, a.patience = patience ? patience : CH_PATIENCE;
  a.eps1 = d->eps1, a.eps2 = d->eps2, a.scale = d->scale * 1.4426950408889634f;
  a.h = h, a.h_out = h_out, a.ldh = ldh;
  a.qkv = words + at[CH_QKV], a.att = words + at[CH_ATTN], a.h1 = words + at[CH_OUT], a.act = words + at[CH_FC], a.h2 = words + at[CH_PROJ];
  a.present = words + at[CH_KINDS];
  a.n_heads = d->n_heads, a.n_kv_heads = d->n_kv_heads, a.q_width = d->n_heads * CH_HEAD, a.kv_width = d->n_kv_heads * CH_HEAD;
  a.page_size = d->page_size, a.page_stride = d->page_stride;
  a.block_table = block_table, a.max_blocks = max_blocks, a.token_req = token_req, a.positions = positions;
  const void* kernel = rows == 1 ? (const void*)decode_chain_kernel<1> : (const void*)decode_chain_kernel<2>;
  // (granted a device at a time: one process may hold engines on several; and always the most, as threads may grant side by side)
  static std::atomic<bool> granted[CH_DEVICES][CHAIN_MOST_ROWS];
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0) FAIL("decode_chain: no current device");
  if (device >= CH_DEVICES || !granted[device][rows - 1]) {
    const int most = CH_LDS_MOST - (int)(rows == 1 ? sizeof(ChainShared<1>) : sizeof(ChainShared<2>));
    hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, most);
    if (e != hipSuccess) FAIL("decode_chain: cannot get %d bytes of LDS: %s", most, hipGetErrorString(e));
    if (device < CH_DEVICES) granted[device][rows - 1] = true;
  }
  hipLaunchKernelGGL(chain_step_kernel, dim3(1), dim3(256), 0, stream, (uint32_t*)memory, (uint32_t)(d->n_layers * CH_KINDS + 1),
                     words + at[0], (int)(n_words - at[0]));
  CHECK_LAUNCH("decode_chain");
  if (rows == 1)
    hipLaunchKernelGGL(decode_chain_kernel<1>, dim3(deal.blocks), dim3(CH_ALL_WAVES * 64), deal.lds, stream, a);
  else
    hipLaunchKernelGGL(decode_chain_kernel<2>, dim3(deal.blocks), dim3(CH_ALL_WAVES * 64), deal.lds, stream, a);
  CHECK_LAUNCH("decode_chain");
  return 0;
}
