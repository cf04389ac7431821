// A row's attention over the keys in its pages, by one block (or, with parts, one of several): the body of the decode
// kernels (attention_decode.hip says how it works and what bounds it) and of the rows that decode beside a prompt's
// portion (attention_prefill.hip).
#pragma once
#include "common.h"
#include "attention_tiles.h"

struct DecodeArgs {
  void* out;  // out, q and the pages hold the kernel's element type
  const void* q;
  const void* k_pages;
  const void* v_pages;
  const int* block_table;
  const int* token_req;
  const int* positions;
  const int* rows;
  float* part_o;
  float* part_ml;
  size_t page_stride;
  int ldq, ldo, max_blocks;
  int n_heads, n_kv_heads, page_size, window, n_splits;
  float scale;
  // Blocks with blockIdx.y >= n_heads have no row: they read `ahead` (chunks of `ahead_pieces`
  // 16-byte pieces: the weights of a product that comes soon) and drop it, each the chunks that
  // a block on its own die will ask for.  Few rows leave most CUs idle, and the memory with them.
  const uint4* ahead;
  size_t ahead_pieces;
  int ahead_chunks;
  // rows_are_requests: item i of `rows` is row i and belongs to request i (a step in which every
  // request brings one token), so neither `rows` nor `token_req` has to be read.
  // table_in_lds: the request's page numbers are copied to LDS once (max_blocks of them fit).
  int rows_are_requests, table_in_lds;
  int page_shift;  // page_size is two to this power, or -1
  int out_head_dim;
  // 1 or 2: the blocks that share a row's keys join their sums themselves: the one that arrives
  // last at the (row, head)'s counter adds them in the order of the parts (no second kernel);
  // 2: n_splits is the most a row takes, and a row takes as many as its own length calls for
  int join_here;
  // Optional terms (all absent: plain causal attention), as in attention.hip's AttnArgs:
  // head_scale [n_heads] instead of `scale`; slopes [n_heads], slope * distance taken off a score;
  // keep_first, the first keys that a window leaves visible; gate (rows of stride ldg, the
  // kernel's element type), the output times its sigmoid.
  const float* head_scale;
  const float* slopes;
  const void* gate;
  int ldg, keep_first;
  // softcap > 0: a scaled score s becomes softcap * tanh(s / softcap); dist_bias [n_heads, n_dist]:
  // dist_bias[h][min(distance, n_dist - 1)] is added to a score
  float softcap;
  const float* dist_bias;
  int n_dist;
  // sinks [n_heads]: exp(sinks[h]) in the softmax's denominator; head_gate (rows of stride ldhg): head
  // h's output times the sigmoid of column h
  const float* sinks;
  const float* head_gate;
  int ldhg;
};

template <typename T>
__device__ __forceinline__ float gate_at(const DecodeArgs& p, int row, int col) {
  if (!p.gate) return 1.f;
  float g;
  if (sizeof(T) == 2)
    g = bits_to_f32(((const uint16_t*)p.gate)[(size_t)row * p.ldg + col]);
  else
    g = ((const float*)p.gate)[(size_t)row * p.ldg + col];
  return 1.0f / (1.0f + expf(-g));
}

#define MAX_WAVES 16

// Sixteen bytes, with the streaming hint where nobody asks for them again
template <bool ONCE>
__device__ __forceinline__ uint4 load16(const void* at) {
  if (!ONCE) return *(const uint4*)at;
  const u32x4_t v = __builtin_nontemporal_load((const u32x4_t*)at);
  return make_uint4(v.x, v.y, v.z, v.w);
}

union Frag8g {
  uint4 u;
  bf16x8_t v;
};

// ldo == 0: out is in the packed order, tiles of 16 rows x 64 columns
__device__ __forceinline__ size_t out_at(const DecodeArgs& p, int row, int col) {
  return p.ldo != 0 ? (size_t)row * p.ldo + col : packed_at(row, col, (p.n_heads * p.out_head_dim + 63) / 64);
}

// What bounds this kernel: the keys and values come from memory once, and at many rows or long contexts that is the
// time (64 rows of 25 heads of 64 at contexts of 300 to 1,001 are 266 MB: 46.7 us, 5.7 TB/s; a plain stream reads 6.4, with
// the streaming hint 7.2).  So they are read with that hint where no two heads share them (8 to 10 % here); a tile is
// small and the next one on its way while it is taken, so that a wave's registers are few and many waves have something
// in flight (tiles of 32 or 64 keys, one at a time, with a lookup and two divisions a lane and key: 54 to 58 us, 13.4 against
// 12.2 for 8 rows, 25.3 against 22.1 for 16 rows of 16 heads of 128, 16.9 against 14.9 for 8 rows of float keys).  At few
// rows and short contexts what is left is the chain: table and query, keys, the waves' join.

// 16 bytes of a row as floats, and a float back as an element
__device__ __forceinline__ void unpack(const uint4& v, float (&f)[8], const uint16_t*) {
  f[0] = __uint_as_float(v.x << 16), f[1] = __uint_as_float(v.x & 0xffff0000u);
  f[2] = __uint_as_float(v.y << 16), f[3] = __uint_as_float(v.y & 0xffff0000u);
  f[4] = __uint_as_float(v.z << 16), f[5] = __uint_as_float(v.z & 0xffff0000u);
  f[6] = __uint_as_float(v.w << 16), f[7] = __uint_as_float(v.w & 0xffff0000u);
}
__device__ __forceinline__ void unpack(const uint4& v, float (&f)[4], const float*) {
  f[0] = __uint_as_float(v.x), f[1] = __uint_as_float(v.y);
  f[2] = __uint_as_float(v.z), f[3] = __uint_as_float(v.w);
}
__device__ __forceinline__ void put(uint16_t* at, float v) { *at = f32_to_bf16_bits(v); }
__device__ __forceinline__ void put(float* at, float v) { *at = v; }

// Joining a row's parts inside the kernel.  The parts' sums pass between blocks on different
// dies, whose L2s do not see each other's lines: they are written and read at agent scope (past
// the die's L2), and a counter a (row, head) says when all are there.  The counters are zero
// between launches (the block that arrives last puts its counter back).
__device__ __forceinline__ void put_shared(float* at, float v) {
  __hip_atomic_store(at, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float get_shared(const float* at) {
  return __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Called by every thread of the block after its put_shared calls; true in all threads of the
// block that arrives last of `n_parts` at `counter`.  No block waits for another.
__device__ __forceinline__ bool last_to_arrive(unsigned* counter, unsigned n_parts, int* s_last) {
  __builtin_amdgcn_s_waitcnt(0);  // this thread's sums have been taken
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned before = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *s_last = before == n_parts - 1;
    if (*s_last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  return *s_last != 0;
}

// (see attn_decode_kernel) The keys of `item`'s head h, part `split` of them, by up to WAVES waves, n_waves of them here.  (The
// caller asks for the block's size, ahead of its branches: asked for here it was one more trip, 0.2 to 0.9 % of a decode step.)
// The launch's dynamic LDS holds max_blocks page numbers with table_in_lds.  PARTS: a row may be in several (p.n_splits);
// join_counters: a counter a (row, head), for parts that are joined here.
template <typename T, int CPK, bool ONCE, bool SHAPED, int WAVES, bool PARTS>
__device__ __forceinline__ void attend_row(const DecodeArgs& p, int wave, int n_waves, int item, int h, int split, unsigned* join_counters) {
  constexpr int EPL = 16 / sizeof(T);  // elements a lane holds of a key
  constexpr int HD = EPL * CPK;
  // two loads of keys at least: where 1 KB holds sixteen keys, a tile of one load left a wave twice the trips (bfloat16,
  // 8 heads of 32, 500 keys, one row: 6.4 us, 5.8 with two loads; 4 rows at 60 to 500 6.5 and 5.9; 16 at 3,000 to 8,000 28.3
  // and 22.7; float, 8 heads of 16, 32 rows at 300 to 1,000 10.2 and 8.7; a row of 50 keys 4.1 and 4.3)
  constexpr int TILE = CPK < 8 ? 2 * ATTN_DECODE_TILE_KEYS : ATTN_DECODE_TILE_KEYS;
  // (keys of 64 bytes a wave has sooner than the parts are joined: one row of 754 keys, float, 12 heads of 16, 6.7 us whole and
  // 7.5 in two parts; bfloat16, 8 heads of 32, 6.8 and 7.6; 4 rows at 512 to 1,000 7.6 and 8.0)
  constexpr int SPLIT_FROM = CPK < 8 ? ATTN_DECODE_SPLIT_KEYS_A_WAVE * 3 / 2 : ATTN_DECODE_SPLIT_KEYS_A_WAVE;
  constexpr int KPL = 64 / CPK;    // keys per load instruction
  constexpr int NL = TILE / KPL;   // loads per tile
  __shared__ float Ms[WAVES], Ls[WAVES];
  __shared__ float Os[WAVES][HD];
  __shared__ int s_last;
  extern __shared__ int page_of[];  // [max_blocks] with table_in_lds

  const int tid = threadIdx.x, lane = tid & 63;
  // Which row, whose pages, at which position: looked up one after the other these are three
  // trips to memory before the first key can be asked for, in a kernel that otherwise makes one
  // or two.  In a decode step item i is row i of request i, and the request's page numbers go to
  // LDS beside the position and the query: one trip, then the keys.
  const int row = p.rows_are_requests ? item : p.rows[item];
  const int req = p.rows_are_requests ? item : p.token_req[row];
  const int kv_head = h / (p.n_heads / p.n_kv_heads);
  const int* table = p.block_table + (size_t)req * p.max_blocks;
  if (p.table_in_lds) {
    const int threads = min((int)blockDim.x, 64 * ATTN_DECODE_ROW_WAVES);  // (the others may be about to end)
    if (tid < threads)
      for (int i = tid; i < p.max_blocks; i += threads) page_of[i] = table[i];
  }
  const int pos = __builtin_amdgcn_readfirstlane(p.positions[row]);
  const int sub = lane % CPK;  // which EPL columns of the key
  const int kin = lane / CPK;  // which key of a load
  const T* k_pages = (const T*)p.k_pages;
  const T* v_pages = (const T*)p.v_pages;

  float qf[EPL];
  {
    const uint4 qv = *(const uint4*)((const T*)p.q + (size_t)row * p.ldq + h * HD + sub * EPL);
    unpack(qv, qf, (const T*)nullptr);
    const float q_scale = p.head_scale ? p.head_scale[h] : p.scale;
#pragma unroll
    for (int i = 0; i < EPL; ++i) qf[i] *= q_scale;
  }
  const float slope = p.slopes ? p.slopes[h] : 0.f;

  const int k_hi = pos + 1;
  const int k_lo = p.window > 0 ? max(0, pos - p.window + 1) : 0;
  // (sixteen waves are for long rows: the others' blocks go on with eight; barriers count the waves that are left)
  if (n_waves > ATTN_DECODE_ROW_WAVES && k_hi - k_lo < ATTN_DECODE_WIDE_ROW_FROM) {
    if (wave >= ATTN_DECODE_ROW_WAVES) return;
    n_waves = ATTN_DECODE_ROW_WAVES;
  }
  const int kt0 = (k_lo / TILE) * TILE;
  // the kept first keys [0, sink_hi) that the window has left behind come first, in tiles of their own
  const int sink_hi = min(p.keep_first, k_lo);
  const int n_sink_tiles = (sink_hi + TILE - 1) / TILE;
  const int n_tiles = n_sink_tiles + (k_hi - kt0 + TILE - 1) / TILE;
  // Joined here, a row may take fewer splits than the launch has: as many as leave a wave
  // ATTN_DECODE_KEYS_A_PART keys, and one if a wave has few anyway (joining costs about 32 keys'
  // time).  Blocks of the splits it does not take have nothing to do.
  int n_splits = PARTS ? p.n_splits : 1;
  if (PARTS && p.join_here == 2) {
    const int keys_a_wave = (k_hi - kt0 + n_sink_tiles * TILE) / n_waves;
    n_splits = keys_a_wave >= SPLIT_FROM ? min(n_splits, keys_a_wave / ATTN_DECODE_KEYS_A_PART) : 1;
    if (split >= n_splits) return;  // (the whole block)
  }
  const int per_split = (n_tiles + n_splits - 1) / n_splits;
  const int t_begin = split * per_split;
  const int t_end = min(n_tiles, t_begin + per_split);

  float m = -INFINITY, l = 0.f, o[EPL];
#pragma unroll
  for (int i = 0; i < EPL; ++i) o[i] = 0.f;

  const size_t head_off = (size_t)kv_head * p.page_size * HD;
  if (p.table_in_lds) __syncthreads();  // (uniform over the block)

  // A tile's loads.  A load's keys lie in one page (a page holds whole loads), so the page, found through scalar
  // arithmetic, is the wave's and only the place within the load a lane's own.  Keys outside the run are pulled
  // inside, loads too (their scores are masked below).
  const int lane_off = kin * HD + sub * EPL;
  auto tile_of = [&](int t, int& kt, int& t_lo, int& t_hi) __attribute__((always_inline)) {
    const bool sink = t < n_sink_tiles;
    kt = sink ? t * TILE : kt0 + (t - n_sink_tiles) * TILE;
    t_lo = sink ? 0 : k_lo, t_hi = sink ? sink_hi : k_hi;  // the run of keys this tile is of
  };
  auto ask = [&](int t, uint4 (&kv)[NL], uint4 (&vv)[NL]) __attribute__((always_inline)) {
    int kt, t_lo, t_hi;
    tile_of(t, kt, t_lo, t_hi);
    const int first = t_lo - t_lo % KPL, last = t_hi - 1 - (t_hi - 1) % KPL;  // the run's first and last load
    const bool whole = kt >= t_lo && kt + TILE <= t_hi;
    int page[NL], in_page[NL];
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      const int b = min(max(kt + j * KPL, first), last);
      const int in_table = p.page_shift >= 0 ? b >> p.page_shift : b / p.page_size;
      in_page[j] = (b - in_table * p.page_size) * HD + (whole ? lane_off : (min(max(b + kin, t_lo), t_hi - 1) - b) * HD + sub * EPL);
      if (p.table_in_lds)  // (pointers that say where they point: one for both would make a flat load)
        page[j] = ((const __attribute__((address_space(3))) int*)page_of)[in_table];
      else
        page[j] = ((const __attribute__((address_space(1))) int*)table)[in_table];
    }
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      const size_t at = (size_t)page[j] * p.page_stride + head_off + in_page[j];
      kv[j] = load16<ONCE>(k_pages + at);
      vv[j] = load16<ONCE>(v_pages + at);
    }
  };
  auto take = [&](int t, const uint4 (&kv)[NL], const uint4 (&vv)[NL]) __attribute__((always_inline)) {
    int kt, t_lo, t_hi;
    tile_of(t, kt, t_lo, t_hi);
    float s[NL];
    float tmax = -INFINITY;
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      float kf[EPL];
      unpack(kv[j], kf, (const T*)nullptr);
      float d = 0.f;
#pragma unroll
      for (int i = 0; i < EPL; ++i) d += qf[i] * kf[i];
      d = group_sum<CPK>(d);  // over the key's lanes
      const int key = kt + j * KPL + kin;
      if (SHAPED && p.softcap > 0.f) d = p.softcap * tanhf(d / p.softcap);
      d -= slope * (float)(pos - key);
      if (SHAPED && p.dist_bias) d += p.dist_bias[(size_t)h * p.n_dist + min(max(pos - key, 0), p.n_dist - 1)];
      s[j] = (key >= t_lo && key < t_hi) ? d : -INFINITY;
      tmax = fmaxf(tmax, s[j]);
    }
    tmax = wave_max(tmax);
    const float m_new = fmaxf(m, tmax);  // finite: every tile holds at least one live key
    const float alpha = __expf(m - m_new);
    l *= alpha;
#pragma unroll
    for (int i = 0; i < EPL; ++i) o[i] *= alpha;
#pragma unroll
    for (int j = 0; j < NL; ++j) {
      const float pj = __expf(s[j] - m_new);  // exp(-inf) = 0 for masked keys
      float vf[EPL];
      unpack(vv[j], vf, (const T*)nullptr);
      if (sub == 0) l += pj;  // one lane of the key's group counts it
#pragma unroll
      for (int i = 0; i < EPL; ++i) o[i] += pj * vf[i];
    }
    m = m_new;
  };
  // the next tile is on its way while one is taken, in two sets of registers by turns
  uint4 k0[NL], v0[NL], k1[NL], v1[NL];
  int t = t_begin + wave;
  if (t < t_end) {
    ask(t, k0, v0);
    for (; t + 2 * n_waves < t_end; t += 2 * n_waves) {
      ask(t + n_waves, k1, v1);
      take(t, k0, v0);
      ask(t + 2 * n_waves, k0, v0);
      take(t + n_waves, k1, v1);
    }
    const bool one_more = t + n_waves < t_end;
    if (one_more) ask(t + n_waves, k1, v1);
    take(t, k0, v0);
    if (one_more) take(t + n_waves, k1, v1);
  }

  // join the lane groups: lanes with the same `sub` hold the same columns
  // (rotations of the row of 16 by 4 and by 8 through DPP moves; rows and halves of the wave
  // through shuffles)
  auto over_groups = [](float v) {
    if (CPK <= 4) v += dpp_move<0x124>(v);  // row_ror:4
    if (CPK <= 8) v += dpp_move<0x128>(v);  // row_ror:8
    if (CPK <= 16) v += __shfl_xor(v, 16, WAVE);
    return v + __shfl_xor(v, 32, WAVE);
  };
  l = over_groups(l);
#pragma unroll
  for (int i = 0; i < EPL; ++i) o[i] = over_groups(o[i]);
  l = group_sum<CPK>(l);

  if (lane == 0) Ms[wave] = m, Ls[wave] = l;
  if (lane < CPK) {
#pragma unroll
    for (int i = 0; i < EPL; ++i) Os[wave][lane * EPL + i] = o[i];
  }
  __syncthreads();

  // every thread joins the waves' results the same way, in the order of the waves
  float M = -INFINITY;
  for (int i = 0; i < n_waves; ++i) M = fmaxf(M, Ms[i]);
  float L = 0.f, acc = 0.f;
  for (int i = 0; i < n_waves; ++i) {
    const float w = (Ms[i] == -INFINITY) ? 0.f : __expf(Ms[i] - M);
    L += Ls[i] * w;
    if (tid < HD) acc += Os[i][tid] * w;
  }
  if (PARTS && n_splits > 1 && p.join_here) {  // (uniform over the block)
    const size_t first = ((size_t)item * p.n_heads + h) * p.n_splits;
    if (tid < HD) put_shared(p.part_o + (first + split) * HD + tid, acc);
    if (tid == 0) put_shared(p.part_ml + (first + split) * 2, M), put_shared(p.part_ml + (first + split) * 2 + 1, L);
    if (!last_to_arrive(join_counters + (size_t)item * p.n_heads + h, (unsigned)n_splits, &s_last)) return;
    if (tid < HD) {  // the parts in their order, whoever arrived when
      float Mj = -INFINITY, Lj = 0.f, aj = 0.f;
      for (int s0 = 0; s0 < n_splits; s0 += 4) {
        float ms[4], ls[4], os[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {  // four parts' values on their way at a time
          const size_t at = first + min(s0 + j, n_splits - 1);
          ms[j] = get_shared(p.part_ml + at * 2), ls[j] = get_shared(p.part_ml + at * 2 + 1);
          os[j] = get_shared(p.part_o + at * HD + tid);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (s0 + j >= n_splits || ms[j] == -INFINITY) continue;  // (a part without a tile)
          const float M2 = fmaxf(Mj, ms[j]);
          const float wa = __expf(Mj - M2), wb = __expf(ms[j] - M2);
          Lj = Lj * wa + ls[j] * wb;
          aj = aj * wa + os[j] * wb;
          Mj = M2;
        }
      }
      put((T*)p.out + out_at(p, row, h * HD + tid),
          aj / with_sink(p, h, Mj, Lj) * head_gate_of(p, row, h) * gate_at<T>(p, row, h * HD + tid));
    }
    return;
  }
  if (tid < HD) {
    if (!PARTS || n_splits == 1) {
      put((T*)p.out + out_at(p, row, h * HD + tid),
          acc / with_sink(p, h, M, L) * head_gate_of(p, row, h) * gate_at<T>(p, row, h * HD + tid));
    } else {
      const size_t base = ((size_t)item * p.n_heads + h) * p.n_splits + split;
      p.part_o[base * HD + tid] = acc;
      if (tid == 0) p.part_ml[base * 2] = M, p.part_ml[base * 2 + 1] = L;
    }
  }
}
