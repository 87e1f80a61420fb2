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
// Two kernels: where the head size is a multiple of 16 up to 128 or 160, 192, 224 or 256, a page holds a multiple of four tokens
// and the pools lie at addresses of that alignment, the tiled one
// on the 32-bit matrix instructions; else one block per (token, head).  Which one is a matter of the model's sizes alone,
// never of the batch.
#include "lds_load.h"
#include "mfma_f32.h"

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
// batch times up to 16 heads of the group.  128 keys at a time (at multiples of 128 of the position): wave w makes the scores
// of keys 16 w .. and 64 + 16 w .. (A operand: keys, straight from the cache, B operand: the rows' queries, kept in registers),
// the waves share the rows' maxima and the exponentials through shared memory, and wave w adds dims 16 (w + 4 i) .. of the
// values (A operand: values, transposed in the page, straight from the cache).  Every key and value is read once a block.
// Lane (r, g) holds, of every 16 x 16 product, column r (a row of the block) and four consecutive keys or dims 4 g + i;
// v_mfma_f32_16x16x4_f32 is full 32-bit, and its operands lie so that scores and outputs are added in the order of channels
// and keys (mfma_f32.h): without a window the results have the bits of the kernel above.  A row's sums never see another
// row: a key it does not see weighs exactly zero and leaves its maximum alone, so how many rows share a tile changes no bit.
// Tokens of several requests in one tile are taken request by request.  A half tile in which some row does not see every key
// and a value is not finite is added key by key by ordinary arithmetic (zero times infinity must not reach a row that does
// not see the key).
// What bounds it: 16 x 128 x hd products of 32-bit twice a tile (1.7 us of the matrix pipe for a block's tile at hd = 128, shared by
// the waves of the other blocks), the ordinary arithmetic beside them and two barriers; keys are on their way while the values before
// them are worked, values while keys are.  The order of the loads is set by registers: at hd = 128 a unit holds two blocks of at most 256
// a lane, with a word more in scratch every tile would wait for all that was just asked for.  500 tokens, 16 heads of 128 over 8 kv
// heads, 32-bit: 46 us, 1000 tokens 122, 8 tokens 12.3 (keys and values of a tile both a tile ahead, 26 words in scratch: 53, 138,
// 14.2; no load sent past a request's last tile, by a condition, behind which the compiler waits for every load: 47, 129, 11.7, but
// 133 for 100 at hd = 256; values asked for when their products were next 62, 177, 13.5); the kernel above, which reads every key
// once per query head with the lanes of a wave hd values apart, took 637.
__device__ __forceinline__ bool finite4(const float4& v) {
  return isfinite(v.x) && isfinite(v.y) && isfinite(v.z) && isfinite(v.w);
}

// Four neighbouring values as they lie in memory, and what becomes of them when they are used.
template <typename T>
struct RawFour {
  typedef float4 type;
  static __device__ __forceinline__ type load(const float* p) { return *reinterpret_cast<const float4*>(p); }
  static __device__ __forceinline__ float4 values(const type& v) { return v; }
  // the first n of them, the others zero
  static __device__ __forceinline__ type first(const type& v, int n) {
    return make_float4(n > 0 ? v.x : 0.f, n > 1 ? v.y : 0.f, n > 2 ? v.z : 0.f, n > 3 ? v.w : 0.f);
  }
};
template <>
struct RawFour<bf16_t> {
  typedef uint2 type;
  static __device__ __forceinline__ type load(const bf16_t* p) { return *reinterpret_cast<const uint2*>(p); }
  static __device__ __forceinline__ float4 values(const type& v) {
    return make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u), __uint_as_float(v.y << 16),
                       __uint_as_float(v.y & 0xffff0000u));
  }
  static __device__ __forceinline__ type first(const type& v, int n) {
    return make_uint2(n > 1 ? v.x : n > 0 ? v.x & 0xffffu : 0u, n > 3 ? v.y : n > 2 ? v.y & 0xffffu : 0u);
  }
};

// hd = 16 KC.  POW2: pages of 2^page_shift keys (a division under a run-time condition would put every load in a block of its own)
template <typename T, int KC, bool POW2>
__global__ void __launch_bounds__(256, KC <= 8 ? 2 : 1)
paged_attention_tiles_kernel(const T* __restrict__ q, int q_stride, T* __restrict__ out, int out_stride,
                             const T* __restrict__ k_pool, const T* __restrict__ v_pool,
                             const int* __restrict__ positions, const int* __restrict__ token_entry,
                             const int* __restrict__ block_table, int bt_stride, int page_size, int page_shift,
                             int T_, int tp, int nq, int nkv, float scale, int window,
                             const float* __restrict__ bias, int bias_rows, const float* __restrict__ sink) {
  constexpr int HD = 16 * KC, NT = (KC + 3) / 4;
  __shared__ float s_max[4][16];
  __shared__ __attribute__((aligned(16))) float s_p[16][132];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
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
  f32x4_t qf[KC];                                        // [c][i]: channel 16 c + 4 i + g
  const T* qp = q + (size_t)t * q_stride + (size_t)h * HD + g;
#pragma unroll
  for (int c = 0; c < KC; ++c)
#pragma unroll
    for (int i = 0; i < 4; ++i) qf[c][i] = ld_f32(qp + 16 * c + 4 * i) * scale;
  f32x4_t acc[NT];
#pragma unroll
  for (int n = 0; n < NT; ++n) acc[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  auto page_index = [&](int j) { return POW2 ? j >> page_shift : j / page_size; };
  auto in_page = [&](int j) { return POW2 ? j & (page_size - 1) : j - j / page_size * page_size; };

  // lane i < n_tok: the block's i-th token
  const int own_entry = token_entry[t0 + (lane < n_tok ? lane : n_tok - 1)], own_pos = positions[t0 + (lane < n_tok ? lane : n_tok - 1)];
  using Raw = RawFour<T>;
  for (int first = 0; first < n_tok;) {
    // the tokens of one request; their last position is the largest, their first one's window starts lowest
    const int seg_entry = __builtin_amdgcn_readlane(own_entry, first);
    const unsigned long long same = __ballot(lane < n_tok && own_entry == seg_entry) >> first;
    const int end = first + __builtin_ctzll(~same);      // n_tok <= 16: some bit above is clear
    const bool inside = lane >= first && lane < end;
    const int hi = -__builtin_amdgcn_readfirstlane(wave_min(inside ? -own_pos : 0x7fffffff));
    const int low = __builtin_amdgcn_readfirstlane(wave_min(inside ? first_seen_key(own_pos, window) : 0x7fffffff));
    const bool alone = first == 0 && end == n_tok;       // no row of the block belongs to another request
    first = end;
    const bool active = valid && entry == seg_entry;
    const int* bt = block_table + (size_t)seg_entry * bt_stride;
    // Keys and values of both halves of a tile.  Up to hd = 128 registers hold three of the four at a time, and the halves' products
    // with the queries alternate: a tile's first keys are asked for before the exponentials of the tile before, its second keys
    // behind the first half of that tile's values, its first values behind the second, its second values when its keys are used up.
    // The entries of the block table they lie by are loaded a tile before them; nothing touches a loaded value or entry until it
    // is used (a select on it would wait for everything on its way).  An entry counts as -1 for keys past the last, and page 0
    // stands in for what has none.
    constexpr int SETS = KC <= 8 ? 2 : 1;
    typename Raw::type kf[SETS][KC], vf[SETS][NT][4];
    int kpage[2], knext[2], vhave[2], vnext[2][4];
    // (relaxed loads, or the compiler moves them down to their use a tile later and waits for all the others there)
    auto entry_of = [&](int j) __attribute__((always_inline)) {
      return __hip_atomic_load(bt + page_index(j <= hi ? j : hi), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
    };
    auto key_entry = [&](int half, int at) __attribute__((always_inline)) { knext[half] = entry_of(at + 64 * half + 16 * wave + r); };
    auto value_entries = [&](int half, int at) __attribute__((always_inline)) {
#pragma unroll
      for (int c = 0; c < 4; ++c) vnext[half][c] = entry_of(at + 64 * half + 16 * c + 4 * g);
    };
    // the keys of half `half` of the tile at `at`, by knext; its page stays in kpage for the tile's tests
    auto fetch_keys = [&](int half, int at) __attribute__((always_inline)) {
      typename Raw::type (&k)[KC] = kf[SETS == 2 ? half : 0];
      const int j = at + 64 * half + 16 * wave + r, page = j <= hi ? knext[half] : -1;
      kpage[half] = page;
      const T* src = k_pool + (((size_t)(page < 0 ? 0 : page) * nkv + kvh) * page_size + (page < 0 ? 0 : in_page(j))) * HD + 4 * g;
#pragma unroll
      for (int c = 0; c < KC; ++c) k[c] = Raw::load(src + 16 * c);
    };
    // half a tile's values for this wave's dims, by vnext; a bit of vhave per chunk: whether the lane's keys of it have a page
    auto fetch_values = [&](int half, int at) __attribute__((always_inline)) {
      typename Raw::type (&v)[NT][4] = vf[SETS == 2 ? half : 0];
      vhave[half] = 0;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int jv = at + 64 * half + 16 * c + 4 * g, page = vnext[half][c];
        const bool have = jv <= hi && page >= 0;
        vhave[half] |= (have ? 1 : 0) << c;
        const T* src = v_pool + ((size_t)(have ? page : 0) * nkv + kvh) * HD * page_size + (have ? in_page(jv) : 0);
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const int dim = 16 * (wave + 4 * n) + r;
          v[n][c] = Raw::load(src + (size_t)(dim < HD ? dim : 0) * page_size);
        }
      }
    };
    int base = low & ~127;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      key_entry(half, base);
      value_entries(half, base);
    }
#pragma unroll
    for (int half = 0; half < SETS; ++half) fetch_keys(half, base);
    fetch_values(0, base);
    // from here on: entries of the half that is fetched next
#pragma unroll
    for (int half = 0; half < SETS; ++half) key_entry(half, base + 128);
    value_entries(0, base + 128);
    for (; base <= hi; base += 128) {
      f32x4_t s[2];
      unsigned long long there[2];                       // bit r: key 16 wave + r of the half has a page
      bool ok[2][4];
      float tile_max = -INFINITY;
      if constexpr (SETS == 2) {
        s[0] = s[1] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < KC; ++c) {
          const f32x4_t k0 = in_order(Raw::values(kf[0][c])), k1 = in_order(Raw::values(kf[1][c]));
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            s[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(k0[i], qf[c][i], s[0], 0, 0, 0);
            s[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(k1[i], qf[c][i], s[1], 0, 0, 0);
          }
        }
      }
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        constexpr bool both = SETS == 2;
        const int at = base + 64 * half;
        if constexpr (!both) {
          s[half] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int c = 0; c < KC; ++c) {
            const f32x4_t k = in_order(Raw::values(kf[0][c]));
#pragma unroll
            for (int i = 0; i < 4; ++i) s[half] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[i], qf[c][i], s[half], 0, 0, 0);
          }
        }
        there[half] = __ballot(kpage[half] >= 0);
        if constexpr (both) {
          if (half == 0) {
            fetch_values(1, base);
            value_entries(1, base + 128);
            fetch_keys(0, base + 128);
            key_entry(0, base + 256);
          }
        } else {
          const int next = half == 0 ? base : base + 128;            // where the other half's next keys lie
          fetch_keys(half ^ 1, next);
          key_entry(half ^ 1, next + 128);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int j = at + 16 * wave + 4 * g + i;
          ok[half][i] = active && j <= pos && j >= lo && ((there[half] >> (4 * g + i)) & 1);
          if (ok[half][i]) tile_max = fmaxf(tile_max, s[half][i]);
        }
      }
      if (bias) {
        tile_max = -INFINITY;
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int j = base + 64 * half + 16 * wave + 4 * g + i;
            if (ok[half][i]) {
              s[half][i] += bias[(size_t)h * bias_rows + (pos - j < bias_rows ? pos - j : bias_rows - 1)];
              tile_max = fmaxf(tile_max, s[half][i]);
            }
          }
      }
      tile_max = max_with_lane_xor32(max_with_lane_xor16(tile_max));
      if (g == 0) s_max[wave][r] = tile_max;
      bare_barrier();                                    // the loads on their way stay on their way
      const float m_new = fmaxf(fmaxf(m, fmaxf(s_max[0][r], s_max[1][r])), fmaxf(s_max[2][r], s_max[3][r]));
      const float alpha = m_new == m ? 1.f : expf(m - m_new);
      // the exponentials lie so that a reader of four neighbouring places has keys g, 4 + g, 8 + g, 12 + g of a chunk
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          s_p[r][64 * half + 16 * wave + 4 * i + g] = ok[half][i] ? expf(s[half][i] - m_new) : 0.f;
      bare_barrier();
      m = m_new;
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[n][i] *= alpha;
      float tile_sum = 0.f;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int at = base + 64 * half;
        constexpr bool both = SETS == 2;
        typename Raw::type (&vh)[NT][4] = vf[both ? half : 0];
        f32x4_t pf[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) pf[c] = *reinterpret_cast<const f32x4_t*>(&s_p[r][64 * half + 16 * c + 4 * g]);
        // the half's sum as a tree over the bits of the key's place, the highest first
        {
          const f32x4_t a = (pf[0] + pf[2]) + (pf[1] + pf[3]);          // [i]: places 4 i + g
          const float sum = (a[0] + a[2]) + (a[1] + a[3]);
          tile_sum += sum_with_lane_xor16(sum_with_lane_xor32(sum));
        }
        // keys past the end and keys without a page count as zero
        if (!__all(vhave[half] == 15 && at + 63 <= hi)) {
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const int left = (vhave[half] >> c) & 1 ? hi - (at + 16 * c + 4 * g) + 1 : 0;
#pragma unroll
            for (int n = 0; n < NT; ++n) vh[n][c] = Raw::first(vh[n][c], left);
          }
        }
        // every row sees every key, or every value is finite
        bool plain = alone && __all(!valid || (at >= lo && at + 63 <= pos));
        if (!plain) {
          bool fine = true;
#pragma unroll
          for (int n = 0; n < NT; ++n)
#pragma unroll
            for (int c = 0; c < 4; ++c) fine = fine && finite4(Raw::values(vh[n][c]));
          plain = __all(fine);
        }
        if (plain) {
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            f32x4_t v[NT];
#pragma unroll
            for (int n = 0; n < NT; ++n) v[n] = in_order(Raw::values(vh[n][c]));
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
              for (int n = 0; n < NT; ++n) acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[n][i], pf[c][i], acc[n], 0, 0, 0);
          }
        } else {
          // lane (r, g) holds dims 4 g + i of row r; the value of key 16 c + 4 o + j at dim 4 g + i lies in lane (4 g + i, o).
          // This rare path must not set the kernel's registers: four keys' values at a time.  For pages that are no power of two it is a
          // loop (written out for every kernel it was half of the family's code, 69 s to compile, now 50), a key at a time, and nothing
          // ahead for all keys: `none` is a zero that the compiler does not see through.
#pragma unroll
          for (int c = 0; c < 4; ++c)
#pragma unroll (POW2 ? 4 : 1)
            for (int o = 0; o < 4; ++o) {
              if constexpr (POW2) __builtin_amdgcn_sched_barrier(0);
              const int have = __shfl(vhave[half], 16 * o, 64);
#pragma unroll
              for (int j = 0; j < 4; ++j) {
                int none = 0;
                if constexpr (!POW2) {
                  __builtin_amdgcn_sched_barrier(0);
#ifdef __HIP_DEVICE_COMPILE__
                  asm volatile("" : "+s"(none));
#endif
                }
                const int key = at + 16 * c + 4 * o + j;
                const bool sees = active && key <= pos && key >= lo && ((have >> c) & 1);
                const float w = s_p[r][64 * half + 16 * c + 4 * j + o + none];
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                  for (int i = 0; i < 4; ++i) {
                    const float4 four = Raw::values(vh[n][c]);
                    const float mine = j == 0 ? four.x : j == 1 ? four.y : j == 2 ? four.z : four.w;
                    const float v = __shfl(mine, 16 * o + 4 * g + i + none, 64);
                    if (sees) acc[n][i] += w * v;
                  }
              }
            }
        }
        if constexpr (both) {
          if (half == 0) {
            fetch_keys(1, base + 128);
            key_entry(1, base + 256);
          } else {
            fetch_values(0, base + 128);
            value_entries(0, base + 256);
          }
        } else {
          const int next = half == 0 ? base : base + 128;
          fetch_values(half ^ 1, next);
          value_entries(half ^ 1, next + 128);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      l = l * alpha + tile_sum;
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
#define AS(KC, POW2) hipLaunchKernelGGL((paged_attention_tiles_kernel<T, KC, POW2>), grid, block, 0, stream, q, q_stride, out, \
    out_stride, k_pool, v_pool, positions, token_entry, block_table, bt_stride, page_size, shift, T_, tp, nq, nkv, scale, \
    window, bias, bias_rows, sink)
#define GO(KC) case KC: if (shift >= 0) AS(KC, true); else AS(KC, false); return true
  switch (hd / 16) {
    GO(1); GO(2); GO(3); GO(4); GO(5); GO(6); GO(7); GO(8); GO(10); GO(12); GO(14); GO(16);
    default: return false;
  }
#undef GO
#undef AS
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
