// What lies between a projection and the attention (or recurrence) that reads its heads, and
// between the attention and the output projection, for mixers that shape their heads in ways of
// their own.  Everything is 32-bit inside; the sources are the projections' float rows.
//
//   (causal convolution)  y[t, c] = sum_j w[c, j] u[t - taps + 1 + j, c] over a request's own tokens;
//                   inputs of earlier steps come from the request's state row ([taps - 1, C], the
//                   latest last, zero at a request's start), which conv_state_update
//                   (linear_state.hip) brings up to date afterwards.  With `conv_single` (every
//                   request brings one token) the kernel moves the state up itself.  It is an
//                   option of head_prepare: the source's columns pass through it on their way in.
//   head_prepare    a wave a (row, head): the head's `dim` columns from a float row (through the
//                   convolution, where one is given); RMS norm over
//                   the first `norm_dim` of them (or, with `norm_whole`, over all heads' columns at
//                   once, with a weight for each) (times a weight of norm_dim values shared by all
//                   heads, or none); rotation of the `rot_dims` columns from `rot_off` on by
//                   position * inv_freq[i], pairs (2i, 2i + 1) or (i, i + rot_dims / 2), cos and
//                   sin times `rot_mult`; then the head goes to `copies` places: copy c of head h
//                   to column dst_head[c * n_heads + h] * dst_stride of the output row (h itself
//                   without a table), zeros from `dim` up to `dst_fill` columns.  The output is
//                   rows of a matrix, or (block_table given) the pages of a cache: the row's
//                   request and position say which page and place, as kv_write has it.
//                   head_prepare_many: up to four such preparations in one launch.
//   diff_combine    o = a1 - lambda a2 per head, where a1 and a2 are two heads of an attention's
//                   output (tables say which), divided by its root mean square and multiplied by
//                   `mult`.
//   head_gate       x[t, h, :] *= sigmoid(g[t, h]), in place, for heads that are there already (the latent attention's gate is a
//                   term of its attention kernels).
#include "common.h"

#define PREPARE_CONV_MAX_DIM 256  // the widest head that passes a convolution

struct PrepareArgs {
  const float* src;
  int lds, src_col, src_stride;  // head h at column src_col + h * src_stride
  int n_rows, n_heads, dim;
  int norm_dim;
  const float* norm_w;  // [norm_dim] or null
  float eps;
  int rot_off, rot_dims, interleaved;
  const float* inv_freq;  // [rot_dims / 2]
  float rot_mult;
  const int* positions;
  void* dst;
  int ldd, dst_stride, dst_fill, copies;
  const int* dst_head;  // [copies, n_heads] or null
  // a causal convolution over the source's columns (column c of the row is channel c), or conv_w null
  const float* conv_w;  // [channels, taps]
  int taps, conv_channels, conv_single;
  float* conv_state;  // a request's row: [taps - 1, channels] at conv_offset, the latest last
  size_t conv_state_stride, conv_offset;
  const int* seq_start;  // [requests] the first row of a request in this step
  const int* slot_ids;   // [requests] its state row
  const int* token_req;  // [rows] (the convolution and the pages need it)
  // dst is a cache's pages (of dst_stride columns a head) where block_table is given
  const int* block_table;
  int max_blocks, page_size;
  size_t page_stride;
  // norm_whole > 0: the norm runs over the whole projection, the norm_whole columns from src_col
  // on (all heads at once), with a weight for every one of them (norm_w [norm_whole]); every
  // column of a head is normed.  Not together with a convolution.
  int norm_whole;
};

template <typename T>
__device__ __forceinline__ void prepare_head(const PrepareArgs& a, long item, int lane) {
  if (item >= (long)a.n_rows * a.n_heads) return;  // whole waves leave; no barrier follows
  const int row = (int)(item / a.n_heads), h = (int)(item % a.n_heads);
  const int first_col = a.src_col + h * a.src_stride;
  const float* s = a.src + (size_t)row * a.lds + first_col;
  const int req = (a.conv_w || a.block_table) ? a.token_req[row] : 0;
  const int local = a.conv_w ? row - a.seq_start[req] : 0;  // the row's place among its request's rows of this step
  float* old = a.conv_w ? a.conv_state + (size_t)a.slot_ids[req] * a.conv_state_stride + a.conv_offset : nullptr;
  // column c of the head as the rest sees it: as it is, or through the convolution (the oldest
  // input first), which is run once a column into the wave's own piece of LDS (the norm, the
  // column's own turn and its partner's read it)
  __shared__ float convolved[4][PREPARE_CONV_MAX_DIM];
  float* cv = convolved[threadIdx.x >> 6];
  if (a.conv_w) {
    for (int c = lane; c < a.dim; c += 64) {
      const int ch = first_col + c;
      float acc = 0.f;
      for (int j = a.taps - 1; j >= 0; --j) {
        const int at = local - j;
        const float u = at >= 0 ? s[c - (long)j * a.lds] : old[(size_t)(a.taps - 1 + at) * a.conv_channels + ch];
        acc += a.conv_w[(size_t)ch * a.taps + (a.taps - 1 - j)] * u;
      }
      cv[c] = acc;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");  // (the wave's lanes read each other's columns)
    __builtin_amdgcn_wave_barrier();
  }
  auto in = [&](int c) { return a.conv_w ? cv[c] : s[c]; };
  float rstd = 1.f;
  if (a.norm_whole > 0) {
    // (every wave of the row adds up the whole projection itself: a few loads a lane)
    const float* whole = a.src + (size_t)row * a.lds + a.src_col;
    float q = 0.f;
    for (int k = lane; k < a.norm_whole; k += 64) q += whole[k] * whole[k];
    rstd = 1.0f / sqrtf(wave_sum(q) / (float)a.norm_whole + a.eps);
  } else if (a.norm_dim > 0) {
    float q = 0.f;
    for (int k = lane; k < a.norm_dim; k += 64) {
      const float u = in(k);
      q += u * u;
    }
    rstd = 1.0f / sqrtf(wave_sum(q) / (float)a.norm_dim + a.eps);
  }
  const int position = (a.rot_dims || a.block_table) ? a.positions[row] : 0;
  const float pos = (float)position;
  const int half = a.rot_dims / 2;
  // where head dh of this row starts in dst
  const size_t page_base = a.block_table ? (size_t)a.block_table[(size_t)req * a.max_blocks + position / a.page_size] * a.page_stride : 0;
  auto head_at = [&](int dh) {
    return a.block_table ? page_base + ((size_t)dh * a.page_size + position % a.page_size) * a.dst_stride
                         : (size_t)row * a.ldd + (size_t)dh * a.dst_stride;
  };
  for (int k = lane; k < a.dst_fill; k += 64) {
    float v = 0.f;
    if (k < a.dim) {
      const int rel = k - a.rot_off;
      auto at = [&](int c) {
        if (a.norm_whole > 0) return in(c) * rstd * (a.norm_w ? a.norm_w[h * a.src_stride + c] : 1.f);
        return c < a.norm_dim ? in(c) * rstd * (a.norm_w ? a.norm_w[c] : 1.f) : in(c);
      };
      v = at(k);
      if (rel >= 0 && rel < a.rot_dims) {
        int i, partner;
        bool first;  // this column is the pair's first member
        if (a.interleaved)
          i = rel >> 1, first = !(rel & 1), partner = first ? k + 1 : k - 1;
        else
          first = rel < half, i = first ? rel : rel - half, partner = first ? k + half : k - half;
        float sn, cs;
        sincosf(pos * a.inv_freq[i], &sn, &cs);
        sn *= a.rot_mult, cs *= a.rot_mult;
        const float other = at(partner);
        v = first ? v * cs - other * sn : v * cs + other * sn;
      }
    }
    for (int c = 0; c < a.copies; ++c) {
      const int dh = a.dst_head ? a.dst_head[c * a.n_heads + h] : h;
      ((T*)a.dst)[head_at(dh) + k] = from_f32<T>(v);
    }
  }
  if (a.conv_w && a.conv_single && a.taps > 1) {
    // every request brings one token: this wave alone reads and writes its request's inputs of this
    // head's channels, so it moves them up by one itself, after everything above has been read
    // (a lane read its neighbours' channels for the rotation: the wave's loads are waited for first)
    __builtin_amdgcn_s_waitcnt(0);
    for (int k = lane; k < a.dim; k += 64) {
      const int ch = first_col + k;
      for (int j = 0; j + 2 < a.taps; ++j) old[(size_t)j * a.conv_channels + ch] = old[(size_t)(j + 1) * a.conv_channels + ch];
      old[(size_t)(a.taps - 2) * a.conv_channels + ch] = s[k];
    }
  }
}

// The same for heads of up to 64 CPL columns, convolutions of up to four taps and norms over a head: what every mixer here
// but those with wider heads or a norm over the whole projection has.  A wave takes R neighbouring rows of a head, one or eight.
//
// What bounds it: at few rows the trips to memory that follow one another, at many rows the same trips, paid once a row and head by
// the kernel above (which looks up a request, its first row, its state row and a page one after another, then takes the
// taps and the norm's weights a load at a time: 1,357 rows of 32 heads of 64 and 8 of 128 through four taps 48 us, 8 rows 8.8; 1,357
// rows of 16 heads of 224 and the latent 18.5).  Here what does not depend on the row's request (the rows with the R + 3 inputs that R outputs
// need, taps, weights, angles) is on its way together with the request and the position, then first row, state row and page
// together, then (only where a request's first rows are among them) the state: 27, 6.4 and 15.5 us.  The sums, and so the bits,
// are those of the kernel above.
#define PREPARE_TAPS 4
template <typename T, int R, int CPL>
__device__ __forceinline__ void prepare_rows(const PrepareArgs& a, int row0, int h, int lane, float* mine) {
  const int first_col = a.src_col + h * a.src_stride;
  const bool conv = a.conv_w != nullptr, pages = a.block_table != nullptr;
  const int back = conv ? a.taps - 1 : 0;  // rows before a row that it needs
  // lane r (of each R) looks things up for row row0 + r
  const int my_row = min(row0 + lane % R, a.n_rows - 1);
  int req = 0, position = 0;
  if (conv || pages) req = a.token_req[my_row];
  if (a.rot_dims || pages) position = a.positions[my_row];
  int col[CPL];
  float u[R + PREPARE_TAPS - 1][CPL], w[PREPARE_TAPS][CPL], weight[CPL], freq[CPL];
#pragma unroll
  for (int c = 0; c < CPL; ++c) col[c] = min(lane + 64 * c, a.dim - 1);  // (columns beyond the head: the last one's values, not used)
#pragma unroll
  for (int i = 0; i < R + PREPARE_TAPS - 1; ++i) {
    if (i < PREPARE_TAPS - 1 - back) continue;  // (uniform)
    const float* s = a.src + (size_t)min(max(row0 - (PREPARE_TAPS - 1) + i, 0), a.n_rows - 1) * a.lds + first_col;
#pragma unroll
    for (int c = 0; c < CPL; ++c) u[i][c] = s[col[c]];
  }
  if (conv)
#pragma unroll
    for (int j = 0; j < PREPARE_TAPS; ++j)
      if (j < a.taps)
#pragma unroll
        for (int c = 0; c < CPL; ++c) w[j][c] = a.conv_w[(size_t)(first_col + col[c]) * a.taps + (a.taps - 1 - j)];
  const int half = a.rot_dims / 2;
#pragma unroll
  for (int c = 0; c < CPL; ++c) {
    weight[c] = a.norm_dim > 0 && a.norm_w ? a.norm_w[min(col[c], a.norm_dim - 1)] : 1.f;
    if (a.rot_dims) {
      const int rel = min(max(col[c] - a.rot_off, 0), a.rot_dims - 1);
      freq[c] = a.inv_freq[a.interleaved ? rel >> 1 : rel < half ? rel : rel - half];
    }
  }
  int local = 0, slot = 0, page = 0;
  if (conv) local = my_row - a.seq_start[req], slot = a.slot_ids[req];
  if (pages) page = a.block_table[(size_t)req * a.max_blocks + position / a.page_size];

  float v[R][CPL];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (!conv) {
#pragma unroll
      for (int c = 0; c < CPL; ++c) v[r][c] = u[PREPARE_TAPS - 1 + r][c];
      continue;
    }
    const int at_start = __builtin_amdgcn_readlane(local, r);  // rows of the request before this one in this step
    float in[PREPARE_TAPS][CPL];
#pragma unroll
    for (int j = 0; j < PREPARE_TAPS; ++j)
#pragma unroll
      for (int c = 0; c < CPL; ++c) in[j][c] = u[PREPARE_TAPS - 1 + r - j][c];
    if (at_start < back) {  // (uniform) inputs of earlier steps, the latest last
      const float* old = a.conv_state + (size_t)__builtin_amdgcn_readlane(slot, r) * a.conv_state_stride + a.conv_offset + first_col;
#pragma unroll
      for (int j = 1; j < PREPARE_TAPS; ++j)
        if (j < a.taps && at_start - j < 0)
#pragma unroll
          for (int c = 0; c < CPL; ++c) in[j][c] = old[(size_t)(back + at_start - j) * a.conv_channels + col[c]];
    }
#pragma unroll
    for (int c = 0; c < CPL; ++c) v[r][c] = 0.f;
#pragma unroll
    for (int j = PREPARE_TAPS - 1; j >= 0; --j)  // the oldest input first
      if (j < a.taps)
#pragma unroll
        for (int c = 0; c < CPL; ++c) v[r][c] += w[j][c] * in[j][c];
  }
  if (a.norm_dim > 0) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      float q = 0.f;
#pragma unroll
      for (int c = 0; c < CPL; ++c)
        if (lane + 64 * c < a.norm_dim) q += v[r][c] * v[r][c];
      const float rstd = 1.0f / sqrtf(wave_sum(q) / (float)a.norm_dim + a.eps);
#pragma unroll
      for (int c = 0; c < CPL; ++c)
        if (lane + 64 * c < a.norm_dim) v[r][c] = v[r][c] * rstd * weight[c];
    }
  }
  if (a.rot_dims) {
    // a column's partner is another lane's: through the wave's own piece of LDS
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int c = 0; c < CPL; ++c) mine[(r * CPL + c) * 64 + lane] = v[r][c];
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      const int k = lane + 64 * c, rel = k - a.rot_off;
      const bool turns = rel >= 0 && rel < a.rot_dims && k < a.dim;
      if (!__any(turns)) continue;
      const bool first = a.interleaved ? !(rel & 1) : rel < half;  // this column is the pair's first member
      const int partner = a.interleaved ? (first ? k + 1 : k - 1) : first ? k + half : k - half;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        float sn, cs;
        sincosf((float)__builtin_amdgcn_readlane(position, r) * freq[c], &sn, &cs);
        sn *= a.rot_mult, cs *= a.rot_mult;
        const float other = mine[r * CPL * 64 + (turns ? partner : k)];
        const float turned = first ? v[r][c] * cs - other * sn : v[r][c] * cs + other * sn;
        v[r][c] = turns ? turned : v[r][c];
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (row0 + r >= a.n_rows) break;
    const int pos = __builtin_amdgcn_readlane(position, r);
    size_t base = (size_t)(row0 + r) * a.ldd, head = a.dst_stride;
    if (pages) {
      base = (size_t)__builtin_amdgcn_readlane(page, r) * a.page_stride + (size_t)(pos % a.page_size) * a.dst_stride;
      head = (size_t)a.page_size * a.dst_stride;
    }
    for (int k = 0; k < a.copies; ++k) {
      T* out = (T*)a.dst + base + (size_t)(a.dst_head ? a.dst_head[k * a.n_heads + h] : h) * head;
#pragma unroll
      for (int c = 0; c < CPL; ++c)
        if (lane + 64 * c < a.dst_fill) out[lane + 64 * c] = from_f32<T>(lane + 64 * c < a.dim ? v[r][c] : 0.f);
    }
  }
  if (R == 1 && conv && a.conv_single && a.taps > 1) {
    // every request brings one token: this wave alone has its request's inputs of this head's channels and moves them up by one
    float* old = a.conv_state + (size_t)__builtin_amdgcn_readlane(slot, 0) * a.conv_state_stride + a.conv_offset + first_col;
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      if (lane + 64 * c >= a.dim) continue;
      float next[PREPARE_TAPS];
#pragma unroll
      for (int j = 0; j + 2 < PREPARE_TAPS; ++j)
        if (j + 2 < a.taps) next[j] = old[(size_t)(j + 1) * a.conv_channels + lane + 64 * c];
#pragma unroll
      for (int j = 0; j + 2 < PREPARE_TAPS; ++j)
        if (j + 2 < a.taps) old[(size_t)j * a.conv_channels + lane + 64 * c] = next[j];
      old[(size_t)(a.taps - 2) * a.conv_channels + lane + 64 * c] = u[PREPARE_TAPS - 1][c];
    }
  }
}
template <typename T, int R>
__device__ __forceinline__ void prepare_any(const PrepareArgs& a, long item, int lane, float* mine) {
  if (item >= (long)((a.n_rows + R - 1) / R) * a.n_heads) return;  // whole waves leave; no barrier follows
  const int row0 = (int)(item / a.n_heads) * R, h = (int)(item % a.n_heads);
  if (a.dst_fill <= 64)
    prepare_rows<T, R, 1>(a, row0, h, lane, mine);
  else if (a.dst_fill <= 128)
    prepare_rows<T, R, 2>(a, row0, h, lane, mine);
  else
    prepare_rows<T, R, 4>(a, row0, h, lane, mine);
}
static bool prepared_in_rows(const PrepareArgs& a) {
  return a.dst_fill <= 256 && a.norm_whole == 0 && (!a.conv_w || a.taps <= PREPARE_TAPS);
}

// Several preparations in one launch (a mixer's queries, keys and values): the blocks of each
// follow those of the one before.
#define PREPARE_MOST 4
struct PrepareMany {
  PrepareArgs seg[PREPARE_MOST];
  unsigned first_block[PREPARE_MOST + 1];
  int n;
};

template <typename T>
__global__ __launch_bounds__(256) void head_prepare_many_kernel(PrepareMany m) {
  int s = 0;
  while (s + 1 < m.n && blockIdx.x >= m.first_block[s + 1]) ++s;
  prepare_head<T>(m.seg[s], (long)(blockIdx.x - m.first_block[s]) * 4 + (threadIdx.x >> 6), threadIdx.x & 63);
}

template <typename T, int R>
__global__ __launch_bounds__(256) void head_prepare_rows_kernel(PrepareMany m) {
  __shared__ float turning[4][R * 256];
  int s = 0;
  while (s + 1 < m.n && blockIdx.x >= m.first_block[s + 1]) ++s;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  prepare_any<T, R>(m.seg[s], (long)(blockIdx.x - m.first_block[s]) * 4 + wave, threadIdx.x & 63, turning[wave]);
}

// A wave a (row, head).
template <typename T>
__global__ __launch_bounds__(256) void diff_combine_kernel(const T* __restrict__ att, int lda, int head_stride,
                                                           const int* __restrict__ first, const int* __restrict__ second,
                                                           float lambda, float mult, float eps, int n_rows, int n_heads,
                                                           int vdim, T* __restrict__ out, int ldo) {
  const int lane = threadIdx.x & 63;
  const long item = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (item >= (long)n_rows * n_heads) return;
  const int row = (int)(item / n_heads), h = (int)(item % n_heads);
  const T* a1 = att + (size_t)row * lda + (size_t)first[h] * head_stride;
  const T* a2 = att + (size_t)row * lda + (size_t)second[h] * head_stride;
  float q = 0.f;
  for (int k = lane; k < vdim; k += 64) {
    const float o = to_f32(a1[k]) - lambda * to_f32(a2[k]);
    q += o * o;
  }
  const float f = mult / sqrtf(wave_sum(q) / (float)vdim + eps);
  for (int k = lane; k < vdim; k += 64)
    out[(size_t)row * ldo + (size_t)h * vdim + k] = from_f32<T>((to_f32(a1[k]) - lambda * to_f32(a2[k])) * f);
}

// Thread (row, column).
template <typename T>
__global__ __launch_bounds__(256) void head_gate_kernel(T* __restrict__ x, int ldx, int head_stride, int n_heads,
                                                        const float* __restrict__ g, int ldg, int n_rows) {
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  const int width = n_heads * head_stride;
  if (e >= (long)n_rows * width) return;
  const int row = (int)(e / width), c = (int)(e % width);
  const float z = g[(size_t)row * ldg + c / head_stride];
  T* p = x + (size_t)row * ldx + c;
  *p = from_f32<T>(to_f32(*p) / (1.0f + expf(-z)));
}

DEFINE_LAST_ERROR(mlxlm_last_error)

static int prepare_args_fit(const PrepareArgs& a) {
  if (!a.src || !a.dst) FAIL("head_prepare: null pointer");
  if (a.dim <= 0 || a.src_col < 0 || a.src_col + (long)(a.n_heads - 1) * a.src_stride + a.dim > a.lds)
    FAIL("head_prepare: %d heads of %d columns, %d apart from column %d, in rows of %d", a.n_heads, a.dim, a.src_stride,
         a.src_col, a.lds);
  if (a.norm_dim < 0 || a.norm_dim > a.dim) FAIL("head_prepare: a norm over %d of %d columns", a.norm_dim, a.dim);
  if (a.norm_whole < 0 || (a.norm_whole > 0 && (a.conv_w || a.norm_whole < (a.n_heads - 1) * a.src_stride + a.dim ||
                                                 a.lds < a.src_col + a.norm_whole)))
    FAIL("head_prepare: a norm over the whole projection of %d columns (no convolution; all heads inside)", a.norm_whole);
  if (a.rot_dims && (a.rot_dims % 2 || a.rot_off < 0 || a.rot_off + a.rot_dims > a.dim || !a.inv_freq || !a.positions))
    FAIL("head_prepare: %d turning columns from %d in a head of %d", a.rot_dims, a.rot_off, a.dim);
  if (a.copies < 1 || a.dst_fill < a.dim || a.dst_fill > a.dst_stride)
    FAIL("head_prepare: %d copies, %d columns filled of %d, a head of %d", a.copies, a.dst_fill, a.dst_stride, a.dim);
  if (!a.block_table && !a.dst_head && (a.copies != 1 || (long)(a.n_heads - 1) * a.dst_stride + a.dst_fill > a.ldd))
    FAIL("head_prepare: the heads do not fit rows of %d", a.ldd);
  if (a.conv_w && a.dim > PREPARE_CONV_MAX_DIM) FAIL("head_prepare: heads of %d columns through a convolution (at most %d)", a.dim, PREPARE_CONV_MAX_DIM);
  if (a.conv_w && (a.taps < 1 || a.conv_channels < a.src_col + (a.n_heads - 1) * a.src_stride + a.dim || !a.conv_state ||
                   !a.seq_start || !a.slot_ids || !a.token_req))
    FAIL("head_prepare: a convolution of %d taps over %d channels needs its state and the rows' requests", a.taps, a.conv_channels);
  if (a.block_table && (!a.token_req || !a.positions || a.max_blocks <= 0 || a.page_size <= 0 || a.dst_fill != a.dst_stride))
    FAIL("head_prepare: pages of %d places need the rows' requests and positions, and whole heads of %d columns", a.page_size, a.dst_stride);
  return 0;
}

// Rows a wave takes where there are many: eight leave a wave's lookups an eighth a row, but its eight rows follow one another
// (norms and turns), 3.5 to 4.5 us of them.  So runs are for launches that give every compute unit several waves of them, eight
// with a convolution, whose inputs a run shares, twelve without.  us, a row and runs of eight, (row, head)s: through four taps 2 heads
// of 64, 2,000 rows (4,000) 4.5 and 7.1, 8,000 (16,000) 11.2 and 9.6; 32 heads, 128 rows (4,096) 4.5 and 7.2, 300 (9,600) 7.0 and
// 8.4, 512 (16,384) 10.2 and 9.3, 2,000 31.1 and 21.0; without, 16 heads of 224, 300 rows (4,800) 5.4 and 8.7, 1,000 (16,000) 11.3 and
// 12.2, 2,000 (32,000) 19.0 and 17.9, 8,000 62 and 48; one head of 224, 128 rows 3.4 and 7.6, 8,000 7.2 and 9.5.
#define PREPARE_ROWS 8
#define PREPARE_RUNS_A_CU 12
#define PREPARE_CONV_RUNS_A_CU 8
template <typename T>
static void launch_many(PrepareMany& m, bool in_rows, hipStream_t stream) {
  bool many = in_rows, conv = false;
  long runs = 0;
  for (int i = 0; i < m.n; ++i) {
    many = many && !(m.seg[i].conv_w && m.seg[i].conv_single);
    conv = conv || m.seg[i].conv_w;
    runs += (long)((m.seg[i].n_rows + PREPARE_ROWS - 1) / PREPARE_ROWS) * m.seg[i].n_heads;
  }
  many = many && runs >= (long)(conv ? PREPARE_CONV_RUNS_A_CU : PREPARE_RUNS_A_CU) * n_compute_units();
  const int R = many ? PREPARE_ROWS : 1;
  unsigned blocks = 0;
  for (int i = 0; i < m.n; ++i) {
    m.first_block[i] = blocks;
    blocks += (unsigned)(((long)((m.seg[i].n_rows + R - 1) / R) * m.seg[i].n_heads + 3) / 4);
  }
  for (int i = m.n; i <= PREPARE_MOST; ++i) m.first_block[i] = blocks;
  if (many)
    hipLaunchKernelGGL((head_prepare_rows_kernel<T, PREPARE_ROWS>), dim3(blocks), dim3(256), 0, stream, m);
  else if (in_rows)
    hipLaunchKernelGGL((head_prepare_rows_kernel<T, 1>), dim3(blocks), dim3(256), 0, stream, m);
  else
    hipLaunchKernelGGL(head_prepare_many_kernel<T>, dim3(blocks), dim3(256), 0, stream, m);
}

// `n` preparations (1 to 4) whose outputs are all of `dst_dtype`, in one launch.
extern "C" int head_prepare_many(const PrepareArgs* args, int n, int dst_dtype, hipStream_t stream) {
  if (n < 1 || n > PREPARE_MOST || !args) FAIL("head_prepare_many: %d preparations (1 to %d)", n, PREPARE_MOST);
  if (dst_dtype != DT_F32 && dst_dtype != DT_BF16) FAIL("head_prepare: unknown dtype code %d", dst_dtype);
  PrepareMany m;
  m.n = 0;
  bool in_rows = true;
  for (int i = 0; i < n; ++i) {
    const PrepareArgs& a = args[i];
    if (a.n_rows <= 0 || a.n_heads <= 0) continue;
    if (prepare_args_fit(a)) return 1;
    in_rows = in_rows && prepared_in_rows(a);
    m.seg[m.n++] = a;
  }
  if (m.n == 0) return 0;
  if (dst_dtype == DT_F32)
    launch_many<float>(m, in_rows, stream);
  else
    launch_many<bf16>(m, in_rows, stream);
  CHECK_LAUNCH("head_prepare_many");
  return 0;
}

extern "C" int head_prepare(const PrepareArgs* args, int dst_dtype, hipStream_t stream) {
  return head_prepare_many(args, 1, dst_dtype, stream);
}

extern "C" int diff_combine(const void* att, int lda, int head_stride, const int* first, const int* second, float lambda,
                            float mult, float eps, int n_rows, int n_heads, int vdim, void* out, int ldo, int dtype,
                            hipStream_t stream) {
  if (n_rows <= 0 || n_heads <= 0) return 0;
  if (!att || !first || !second || !out) FAIL("diff_combine: null pointer");
  if (vdim <= 0 || vdim > head_stride || ldo < n_heads * vdim) FAIL("diff_combine: values of %d in heads of %d, rows of %d", vdim, head_stride, ldo);
  if (dtype != DT_F32 && dtype != DT_BF16) FAIL("diff_combine: unknown dtype code %d", dtype);
  const long items = (long)n_rows * n_heads;
  dim3 grid((unsigned)((items + 3) / 4)), block(256);
  if (dtype == DT_F32)
    hipLaunchKernelGGL(diff_combine_kernel<float>, grid, block, 0, stream, (const float*)att, lda, head_stride, first, second,
                       lambda, mult, eps, n_rows, n_heads, vdim, (float*)out, ldo);
  else
    hipLaunchKernelGGL(diff_combine_kernel<bf16>, grid, block, 0, stream, (const bf16*)att, lda, head_stride, first, second,
                       lambda, mult, eps, n_rows, n_heads, vdim, (bf16*)out, ldo);
  CHECK_LAUNCH("diff_combine");
  return 0;
}

extern "C" int head_gate(void* x, int ldx, int head_stride, int n_heads, const float* g, int ldg, int n_rows, int dtype,
                         hipStream_t stream) {
  if (n_rows <= 0 || n_heads <= 0) return 0;
  if (!x || !g) FAIL("head_gate: null pointer");
  if (head_stride <= 0 || ldx < n_heads * head_stride || ldg < n_heads)
    FAIL("head_gate: %d heads of %d columns in rows of %d, gates in rows of %d", n_heads, head_stride, ldx, ldg);
  if (dtype != DT_F32 && dtype != DT_BF16) FAIL("head_gate: unknown dtype code %d", dtype);
  const long total = (long)n_rows * n_heads * head_stride;
  dim3 grid((unsigned)((total + 255) / 256)), block(256);
  if (dtype == DT_F32)
    hipLaunchKernelGGL(head_gate_kernel<float>, grid, block, 0, stream, (float*)x, ldx, head_stride, n_heads, g, ldg, n_rows);
  else
    hipLaunchKernelGGL(head_gate_kernel<bf16>, grid, block, 0, stream, (bf16*)x, ldx, head_stride, n_heads, g, ldg, n_rows);
  CHECK_LAUNCH("head_gate");
  return 0;
}
