// Paged grouped-query attention, general form: any head size up to 1024, any number of heads and
// groups, any page size, any mix of prompt portions and single decoded tokens, optional window or chunk (a negative `window`).
// Keys are visited in tiles in a fixed order that depends only on the token's own position, so the
// result for a token is the same however the batch was cut.  Scores, running maximum, sum and output are 32-bit.  Optionally a bias by
// distance is added to every score: bias[head, min(query position - key position, bias_rows - 1)]
// (float32 [nq, bias_rows]); the scale does not multiply it.  Optionally a sink per head (float32 [nq]): one more
// term exp(sink[head]) in the softmax's denominator that has no key and no value and is not scaled.
// Pools: keys [page, kv_head, row, head_dim]; values [page, kv_head, head_dim, row].
//
// Semantics as the reference asks of its attention library (ullm/layers/attention.py:76-104,
// 298-309): scale = given (head_dim^-0.5, ullm/models/qwen3.py:81), causal with the queries at the
// end of the keys, query head h reads kv head h / (nq / nkv).
//
// Two kernels: where the head size is a multiple of 16 up to 256 and a page holds a multiple of four tokens, the tiled one
// on the 32-bit matrix instructions; else one block per (token, head).  Which one is a matter of the model's sizes alone,
// never of the batch.
#include "common.h"

#define ATT_THREADS 128
#define ATT_MAX_HD 1024

template <typename T>
__global__ void __launch_bounds__(ATT_THREADS)
paged_attention_generic_kernel(const T* __restrict__ q, int q_stride, T* __restrict__ out, int out_stride,
                               const T* __restrict__ k_pool, const T* __restrict__ v_pool,
                               const int* __restrict__ positions, const int* __restrict__ token_entry,
                               const int* __restrict__ block_table, int bt_stride, int page_size,
                               int nq, int nkv, int hd, float scale, int window,
                               const float* __restrict__ bias, int bias_rows,
                               const float* __restrict__ sink) {
  __shared__ float q_s[ATT_MAX_HD];
  __shared__ float p_s[ATT_THREADS];
  __shared__ long long row_s[ATT_THREADS];
  __shared__ float scratch[16];
  const int t = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int kvh = h / (nq / nkv);
  const int pos = positions[t];
  const int* bt = block_table + (size_t)token_entry[t] * bt_stride;
  const int lo = first_seen_key(pos, window);
  const int hi = pos;
  const T* qp = q + (size_t)t * q_stride + (size_t)h * hd;
  for (int i = tid; i < hd; i += ATT_THREADS) q_s[i] = ld_f32(qp + i) * scale;
  __syncthreads();

  constexpr int DPT = ATT_MAX_HD / ATT_THREADS;  // output dims per thread
  float acc[DPT];
#pragma unroll
  for (int r = 0; r < DPT; ++r) acc[r] = 0.f;
  float m = -INFINITY, l = 0.f;

  for (int base = lo; base <= hi; base += ATT_THREADS) {
    const int j = base + tid;
    float s = -INFINITY;
    long long row = -1;
    if (j <= hi) {
      const int page = bt[j / page_size];
      if (page >= 0) {
        row = ((long long)page * nkv + kvh) * page_size + (j % page_size);
        const T* kp = k_pool + row * hd;
        float d = 0.f;
        for (int i = 0; i < hd; ++i) d += q_s[i] * ld_f32(kp + i);
        // a learned bias by distance: one row of the table per head, the last entry for every greater distance
        if (bias) d += bias[(size_t)h * bias_rows + (pos - j < bias_rows ? pos - j : bias_rows - 1)];
        s = d;
      }
    }
    const float tile_max = block_max(s, scratch);
    const float m_new = fmaxf(m, tile_max);
    // the token's own key is always present, so m_new is finite from the first tile that holds it;
    // a tile without any valid key leaves everything unchanged
    const float p = (row >= 0) ? expf(s - m_new) : 0.f;
    const float tile_sum = block_sum(p, scratch);
    __syncthreads();
    p_s[tid] = p;
    row_s[tid] = row;
    __syncthreads();
    const float alpha = (m == -INFINITY) ? 0.f : expf(m - m_new);
    l = l * alpha + tile_sum;
    const int n_tile = (hi - base + 1 < ATT_THREADS) ? hi - base + 1 : ATT_THREADS;
#pragma unroll
    for (int r = 0; r < DPT; ++r) {
      const int d = tid + r * ATT_THREADS;
      if (d < hd) {
        float a = acc[r] * alpha;
        for (int jj = 0; jj < n_tile; ++jj) {
          const long long vr = row_s[jj];
          if (vr >= 0) a += p_s[jj] * ld_f32(v_pool + (vr / page_size) * page_size * hd + (size_t)d * page_size + vr % page_size);
        }
        acc[r] = a;
      }
    }
    if (m_new > -INFINITY) m = m_new;
  }
  T* op = out + (size_t)t * out_stride + (size_t)h * hd;
  float keep = 1.f;
  if (sink) {
    // the sink joins the denominator alone: sum and outputs move to the larger of the two reference values
    const float sv = sink[h];
    const float m_all = fmaxf(m, sv);
    keep = (m == -INFINITY) ? 0.f : expf(m - m_all);
    l = l * keep + expf(sv - m_all);
  }
  const float inv = l > 0.f ? keep / l : 0.f;
#pragma unroll
  for (int r = 0; r < DPT; ++r) {
    const int d = tid + r * ATT_THREADS;
    if (d < hd) st_f32(op + d, acc[r] * inv);
  }
}

// ------------------------------------------------------------------------------- tiles on the 32-bit matrix cores
// A block of four waves takes 16 rows, a row being a (token, query head) pair of one kv head: `tp` consecutive tokens of the
// batch times up to 16 heads of the group.  64 keys at a time (at multiples of 64 of the position): wave w makes the scores
// of keys 16w .. 16w + 15 (A operand: keys, straight from the cache, B operand: the rows' queries, kept in registers), the
// waves share the rows' maxima and the exponentials through shared memory, and wave w adds dims 16 (w + 4i) .. of the
// values (A operand: values, transposed in the page, straight from the cache).  Every key and value is read once a block.
// Lane (r, g) holds, of every 16 x 16 product, column r (a row of the block) and four consecutive keys or dims 4g + i;
// v_mfma_f32_16x16x4_f32 is full 32-bit.  A row's sums never see another row: a key it does not see weighs exactly zero and
// leaves its maximum alone, so how many rows share a tile changes no bit.  Tokens of several requests in one tile are taken
// request by request.  A tile in which some row does not see every key and a value is not finite is added key by key by
// ordinary arithmetic (zero times infinity must not reach a row that does not see the key).
// What bounds it: 16 x 64 x hd products of 32-bit twice a tile (1.7 us of the matrix pipe for a block at hd = 128, shared by
// the waves of the other blocks) and two barriers; the keys of the next tile are on their way while this one's exponentials
// and values are worked.  500 tokens, 16 heads of 128 over 8 kv heads, 32-bit: 55 us; the kernel above, which reads every
// key once per query head with the lanes of a wave hd values apart, took 637.
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
__device__ __forceinline__ float4 ld4_f32(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 ld4_f32(const bf16_t* p) {
  const uint2 u = *reinterpret_cast<const uint2*>(p);
  return make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                     __uint_as_float(u.y & 0xffff0000u));
}
__device__ __forceinline__ float at4(const float4& v, int j) { return j == 0 ? v.x : j == 1 ? v.y : j == 2 ? v.z : v.w; }
__device__ __forceinline__ bool finite4(const float4& v) {
  return isfinite(v.x) && isfinite(v.y) && isfinite(v.z) && isfinite(v.w);
}

template <typename T, int KC>                     // hd = 16 KC
__global__ void __launch_bounds__(256)
paged_attention_tiles_kernel(const T* __restrict__ q, int q_stride, T* __restrict__ out, int out_stride,
                             const T* __restrict__ k_pool, const T* __restrict__ v_pool,
                             const int* __restrict__ positions, const int* __restrict__ token_entry,
                             const int* __restrict__ block_table, int bt_stride, int page_size, int page_shift,
                             int T_, int tp, int nq, int nkv, float scale, int window,
                             const float* __restrict__ bias, int bias_rows, const float* __restrict__ sink) {
  constexpr int HD = 16 * KC, NT = (KC + 3) / 4;
  __shared__ float s_max[4][16], s_sum[4][16];
  __shared__ __attribute__((aligned(16))) float s_p[16][68];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, g = lane >> 4;
  const int group = nq / nkv, gh = group < 16 ? group : 16, chunks = (group + 15) / 16;
  const int kvh = blockIdx.y / chunks, h0 = blockIdx.y % chunks * 16;
  const int t0 = ((int)gridDim.x - 1 - (int)blockIdx.x) * tp;          // later tokens see more keys: they start first
  const int n_tok = T_ - t0 < tp ? T_ - t0 : tp;
  // this lane's row
  const int tt = r / gh, hh = h0 + r % gh;
  const bool valid = tt < n_tok && hh < group;
  const int t = t0 + (tt < n_tok ? tt : 0), h = kvh * group + (hh < group ? hh : 0);
  const int pos = positions[t], entry = token_entry[t];
  const int lo = first_seen_key(pos, window);
  float4 qf[KC];
  const T* qp = q + (size_t)t * q_stride + (size_t)h * HD + 4 * g;
#pragma unroll
  for (int c = 0; c < KC; ++c)
    qf[c] = make_float4(ld_f32(qp + 16 * c) * scale, ld_f32(qp + 16 * c + 1) * scale, ld_f32(qp + 16 * c + 2) * scale,
                        ld_f32(qp + 16 * c + 3) * scale);
  f32x4_t acc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  auto page_index = [&](int j) { return page_shift >= 0 ? j >> page_shift : j / page_size; };

  for (int first = 0; first < n_tok;) {
    // the tokens of one request; their last position is the largest, their first one's window starts lowest
    const int seg_entry = token_entry[t0 + first];
    int end = first, hi = -1, low = 0x7fffffff;
    while (end < n_tok && token_entry[t0 + end] == seg_entry) {
      const int p = positions[t0 + end], f = first_seen_key(p, window);
      hi = p > hi ? p : hi;
      low = f < low ? f : low;
      ++end;
    }
    const bool alone = first == 0 && end == n_tok;       // no row of the block belongs to another request
    first = end;
    const bool active = valid && entry == seg_entry;
    const int* bt = block_table + (size_t)seg_entry * bt_stride;
    int base = low & ~63;
    // pages of a tile: of this lane's key for the scores, of its four keys of every 16 for the values
    int kpage, vpage[4];
    auto pages_of = [&](int at, int& kp, int* vp) __attribute__((always_inline)) {
      const int j = at + 16 * wave + r;
      const int kv = bt[page_index(j <= hi ? j : hi)];
      kp = j <= hi ? kv : -1;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int jv = at + 16 * c + 4 * g;
        const int pv = bt[page_index(jv <= hi ? jv : hi)];
        vp[c] = jv <= hi ? pv : -1;
      }
    };
    float4 kf[KC];
    auto fetch_keys = [&](int at, int kp) __attribute__((always_inline)) {
      const int j = at + 16 * wave + r;
      const T* src = k_pool + (((size_t)(kp < 0 ? 0 : kp) * nkv + kvh) * page_size + (kp < 0 ? 0 : j - page_index(j) * page_size)) * HD + 4 * g;
#pragma unroll
      for (int c = 0; c < KC; ++c) kf[c] = ld4_f32(src + 16 * c);
    };
    pages_of(base, kpage, vpage);
    fetch_keys(base, kpage);
    for (; base <= hi; base += 64) {
      const unsigned long long there = __ballot(kpage >= 0);            // bit r: key 16 wave + r has a page
      float4 vf[NT][4];
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        const int dim = 16 * (wave + 4 * n) + r;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const int jv = base + 16 * c + 4 * g;
          const bool have = vpage[c] >= 0;
          const size_t row = ((size_t)(have ? vpage[c] : 0) * nkv + kvh) * HD + (dim < HD ? dim : 0);
          vf[n][c] = ld4_f32(v_pool + row * page_size + (have ? jv - page_index(jv) * page_size : 0));
          // keys past the end, or without a page, have no value
          if (!have) vf[n][c].x = 0.f;
          if (!have || jv + 1 > hi) vf[n][c].y = 0.f;
          if (!have || jv + 2 > hi) vf[n][c].z = 0.f;
          if (!have || jv + 3 > hi) vf[n][c].w = 0.f;
        }
      }
      int vhave = 0;
#pragma unroll
      for (int c = 0; c < 4; ++c) vhave |= (vpage[c] >= 0 ? 1 : 0) << c;
      f32x4_t sc = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < KC; ++c)
#pragma unroll
        for (int j = 0; j < 4; ++j) sc = __builtin_amdgcn_mfma_f32_16x16x4f32(at4(kf[c], j), at4(qf[c], j), sc, 0, 0, 0);
      pages_of(base + 64, kpage, vpage);                 // clamped to the last key's page past the end
      fetch_keys(base + 64, kpage);
      float s[4], tile_max = -INFINITY;
      bool ok[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = base + 16 * wave + 4 * g + i;
        ok[i] = active && j <= pos && j >= lo && ((there >> (4 * g + i)) & 1);
        s[i] = sc[i];
        if (bias && ok[i]) s[i] += bias[(size_t)h * bias_rows + (pos - j < bias_rows ? pos - j : bias_rows - 1)];
        if (ok[i]) tile_max = fmaxf(tile_max, s[i]);
      }
      tile_max = max_with_lane_xor32(max_with_lane_xor16(tile_max));
      if (g == 0) s_max[wave][r] = tile_max;
      __syncthreads();
      const float m_new = fmaxf(fmaxf(m, fmaxf(s_max[0][r], s_max[1][r])), fmaxf(s_max[2][r], s_max[3][r]));
      const float alpha = m_new == m ? 1.f : expf(m - m_new);
      float p[4], sum = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[i] = ok[i] ? expf(s[i] - m_new) : 0.f;
        sum += p[i];
      }
      *reinterpret_cast<float4*>(&s_p[r][16 * wave + 4 * g]) = make_float4(p[0], p[1], p[2], p[3]);
      sum += __shfl_xor(sum, 16, 64);
      sum += __shfl_xor(sum, 32, 64);
      if (g == 0) s_sum[wave][r] = sum;
      __syncthreads();
      l = l * alpha + ((s_sum[0][r] + s_sum[1][r]) + (s_sum[2][r] + s_sum[3][r]));
      m = m_new;
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[n][i] *= alpha;
      // every row sees every key, or every value is finite
      bool plain = alone && __all(!valid || (base >= lo && base + 63 <= pos));
      if (!plain) {
        bool fine = true;
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
          for (int c = 0; c < 4; ++c) fine = fine && finite4(vf[n][c]);
        plain = __all(fine);
      }
      if (plain) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const float4 pf = *reinterpret_cast<const float4*>(&s_p[r][16 * c + 4 * g]);
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int n = 0; n < NT; ++n)
              acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(at4(vf[n][c], j), at4(pf, j), acc[n], 0, 0, 0);
        }
      } else {
        // lane (r, g) holds dims 4g + i of row r; the value of key 16c + 4o + j at dim 4g + i lies in lane (4g + i, o)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          for (int o = 0; o < 4; ++o) {
            const int have = __shfl(vhave, 16 * o, 64);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const int key = base + 16 * c + 4 * o + j;
              const bool sees = active && key <= pos && key >= lo && ((have >> c) & 1);
              const float w = s_p[r][16 * c + 4 * o + j];
#pragma unroll
              for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                  const float v = __shfl(at4(vf[n][c], j), 16 * o + 4 * g + i, 64);
                  if (sees) acc[n][i] += w * v;
                }
            }
          }
      }
    }
    __syncthreads();                                     // the next request's maxima are written only now
  }
  float keep = 1.f;
  if (sink) {
    const float sv = sink[h];
    const float m_all = fmaxf(m, sv);
    keep = (m == -INFINITY) ? 0.f : expf(m - m_all);
    l = l * keep + expf(sv - m_all);
  }
  const float inv = l > 0.f ? keep / l : 0.f;
  if (!valid) return;
#pragma unroll
  for (int n = 0; n < NT; ++n) {
    const int dim = 16 * (wave + 4 * n) + 4 * g;
    if (dim >= HD) continue;
    T* op = out + (size_t)t * out_stride + (size_t)h * HD + dim;
#pragma unroll
    for (int i = 0; i < 4; ++i) st_f32(op + i, acc[n][i] * inv);
  }
}

// single: no two tokens of the batch belong to one request (each then has a block of its own per kv head)
template <typename T>
static bool launch_tiles(const T* q, int q_stride, T* out, int out_stride, const T* k_pool, const T* v_pool,
                         const int* positions, const int* token_entry, const int* block_table, int bt_stride, int page_size,
                         int T_, int nq, int nkv, int hd, float scale, int window, const float* bias, int bias_rows,
                         const float* sink, int single, hipStream_t stream) {
  const uintptr_t align = sizeof(T) == 4 ? 15 : 7;
  if (hd % 16 || page_size % 4 || ((uintptr_t)k_pool & align) || ((uintptr_t)v_pool & align)) return false;
  const int group = nq / nkv, chunks = (group + 15) / 16, tp = single ? 1 : 16 / (group < 16 ? group : 16);
  int shift = -1;
  for (int b = 2; b < 31; ++b)
    if (page_size == 1 << b) shift = b;
  if ((long long)nkv * chunks > 65535) return false;
  dim3 grid((T_ + tp - 1) / tp, nkv * chunks), block(256);
#define GO(KC) case KC: hipLaunchKernelGGL((paged_attention_tiles_kernel<T, KC>), grid, block, 0, stream, q, q_stride, out, \
    out_stride, k_pool, v_pool, positions, token_entry, block_table, bt_stride, page_size, shift, T_, tp, nq, nkv, scale, \
    window, bias, bias_rows, sink); return true
  switch (hd / 16) {
    GO(1); GO(2); GO(3); GO(4); GO(5); GO(6); GO(7); GO(8); GO(10); GO(12); GO(14); GO(16);
    default: return false;
  }
#undef GO
}

extern "C" int ullm_paged_attention_generic(
    const void* q, int q_stride, void* out, int out_stride, const void* k_pool, const void* v_pool,
    const int* positions, const int* token_entry, const int* block_table, int bt_stride, int page_size,
    int T_, int nq, int nkv, int hd, float scale, int window, const float* bias, int bias_rows,
    const float* sink, int single, int dtype, hipStream_t stream) {
  if (T_ <= 0) return 0;
  if (bias && bias_rows <= 0) return ULLM_ERR_SHAPE;
  if (hd <= 0 || hd > ATT_MAX_HD || nq <= 0 || nkv <= 0 || nq % nkv != 0 || page_size <= 0)
    return ULLM_ERR_SHAPE;
#define TILES(TT) launch_tiles<TT>((const TT*)q, q_stride, (TT*)out, out_stride, (const TT*)k_pool, (const TT*)v_pool, positions, \
    token_entry, block_table, bt_stride, page_size, T_, nq, nkv, hd, scale, window, bias, bias_rows, sink, single, stream)
  if (dtype == ULLM_F32 ? TILES(float) : dtype == ULLM_BF16 && TILES(bf16_t)) ULLM_LAUNCH_CHECK();
#undef TILES
  dim3 grid(T_, nq), block(ATT_THREADS);
#define GO(TT) hipLaunchKernelGGL(paged_attention_generic_kernel<TT>, grid, block, 0, stream, \
    (const TT*)q, q_stride, (TT*)out, out_stride, (const TT*)k_pool, (const TT*)v_pool, positions, \
    token_entry, block_table, bt_stride, page_size, nq, nkv, hd, scale, window, bias, bias_rows, sink)
  if (dtype == ULLM_F32) GO(float);
  else if (dtype == ULLM_BF16) GO(bf16_t);
  else return ULLM_ERR_DTYPE;
#undef GO
  ULLM_LAUNCH_CHECK();
}
