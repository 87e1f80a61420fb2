// out = x W^T in bfloat16 for 17 to 1024 rows where one round of blocks holds them (beyond 1024 only where launches take the time): x [M, K], W [N, K] as the
// reference stores its linears' weights (ullm/layers/linear.py:165,268).
//   store   bfloat16 [M, N], with an optional bias and activation
//   gated   W holds gate rows, then as many up rows: bfloat16 [M, N / 2] of silu(gate) * up (or the clamped unit)
//   float   the 32-bit sums, [slices, M, N]: K is cut into slices, each with a sum of its own, where the matrix alone gives too
//           few blocks for the chip.  Who adds them is the caller's business (the add + norm kernel does, in order)
//
// At these row counts the product is a read of W and a handful of tiles a compute unit, and its time is what a block takes to
// walk its K: so a block's tile (its shape below) is as large as still gives every compute unit one, and the shape and the slices
// are picked by the time they are estimated to take (ullm_gemm_panels_plan).  Operands go straight to shared memory (lds_load.h),
// several stages of 64 values of K on their way: rows of 128 bytes whose 16-byte piece c of row r lies at piece c ^ ((r >> 1) & 7)
// (the 16 lanes that shared memory serves together then read 16 different bank groups), 8 rows an instruction.  Loads of W do
// not stay in the caches, x's do: without that 64 rows of gate|up 24576 x 4096 take 42 us instead of 36.  Blocks of different
// columns begin at different stages of K (block column b at stage b, around the end to the beginning): rows that lie a power of two apart
// otherwise ask the same memory channels at the same time (64 rows 42.5 -> 35.0 us, 130 rows 50.6 -> 45.4).
//
// Two kernels share this:
//   panels    the waves of a block share its stages, each takes TM x TN products of 16 x 16; one barrier a stage, operands of
//             one half of a stage read between the products of the half before.  For tiles of 96 x 64 up to 256 x 128
//   quarters  four waves, each with the whole tile, a quarter of the block's K and stages of its own: no barrier, half the reads of
//             shared memory a product, and a quarter as many stages one after the other; the four sums meet in shared memory at
//             the end.  For tiles of 32 x 16 up to 64 x 96, what small matrices and few rows leave a compute unit
//
// Measured alone (inside a step some 5 % more: gate|up of 130 rows 49) against the kernels that took these calls before, us (cold weights): gate|up 24576 x 4096 17 / 32 / 64 / 130 / 256 rows
// 36 / 38 / 43 / 62 / 69 -> 32 / 33 / 36 / 46 / 58 (130 on: the library and the activation kernel), 6144 x 1024 40 / 130 / 256 / 512 /
// 800 rows 7.9 / 11.6 / 15.1 / 16.4 / 17.3 -> 5.8 / 8.4 / 9.6 / 12.7 / 15.0; partial sums of 4096 x 12288 130 / 256 / 512 rows 31 / 42 / 83
// -> 26 / 36 / 51, of 4096 x 4096 12.9 / 19.4 / 30.0 -> 13.8 / 17 / 24 (at 130 rows with the norm that adds them 21.8 -> 18.1); 1024 x 2048 256 / 512 rows 8.6 / 9.5 -> 6.3 / 7.8.  What bounds them at few
// rows is W (201 MB at 64 rows 5.6 TB/s), else what the second-level caches deliver: every shape gets 64 KB a us and compute
// unit of them, 16 TB/s in all, and the larger a tile the more products it makes of that; around it a launch, the first loads' way
// and the store, 2 to 7 us.
#include "mfma_tiles.h"
#include "launchers.h"

enum { PANELS_STORE = 0, PANELS_GATED = 1, PANELS_FLOAT = 2 };

struct PanelsArgs {
  const bf16_t* x;
  int ldx;
  const bf16_t* w;
  int ldw;
  const float* bias;
  void* out;
  int ldo;
  int M, N, stages, slices, m_tiles, n_tiles;      // N: rows of W; stages: K / 64
  float limit, alpha;
  int act;
};

// A block's work: rows m0 .. of x, output columns n0 .. (gated: gate and up rows of them), stages first .. first + steps of K.
struct PanelsItem {
  int m0, n0, column, slice;
  bool any;
};

// Blocks go to the chip's 8 dies round-robin by their id and every die has a second-level cache of its own: die d takes the d-th
// eighth of the items, slice by slice, up to eight tiles of rows to a strip of W and strip after strip.
__device__ __forceinline__ PanelsItem panels_item(const PanelsArgs& a, int rows, int cols) {
  const int per_slice = a.m_tiles * a.n_tiles, total = per_slice * a.slices, per_die = (total + 7) / 8;
  const int item = ((int)blockIdx.x & 7) * per_die + ((int)blockIdx.x >> 3);
  const bool any = (int)(blockIdx.x >> 3) < per_die && item < total;
  const int slice = item / per_slice, in_slice = item - slice * per_slice;
  const int band = in_slice / (8 * a.n_tiles), in_band = in_slice - band * 8 * a.n_tiles;
  const int high = a.m_tiles - 8 * band < 8 ? a.m_tiles - 8 * band : 8;
  const int column = in_band / (high > 0 ? high : 1);
  return PanelsItem{(8 * band + in_band - column * high) * rows, column * cols, column, slice, any};
}

// Row j of the panel of W that a block of COLS output columns reads, in units of W's rows; gated: HALF columns' gate rows, then
// their up rows, HALF by HALF (a wave's own columns).
template <bool GATED, int HALF>
__device__ __forceinline__ int panels_w_row(const PanelsArgs& a, int n0, int j) {
  if (!GATED) {
    const int n = n0 + j;
    return n < a.N ? n : a.N - 1;
  }
  const int n_out = a.N >> 1, group = j / (2 * HALF), t = j - group * 2 * HALF;
  const bool up = t >= HALF;
  const int n = n0 + group * HALF + (up ? t - HALF : t);
  return (up ? n_out : 0) + (n < n_out ? n : n_out - 1);
}

// Four neighbouring columns c .. c + 3 of one row on their way out (v: the sums; up: the up half's).
template <int MODE>
__device__ __forceinline__ float4 panels_finish(const PanelsArgs& a, float4 v, const float4& up, int c) {
  if (MODE == PANELS_GATED)
    return make_float4(gated_unit(v.x, up.x, a.limit, a.alpha), gated_unit(v.y, up.y, a.limit, a.alpha),
                       gated_unit(v.z, up.z, a.limit, a.alpha), gated_unit(v.w, up.w, a.limit, a.alpha));
  if (MODE == PANELS_STORE) {
    if (a.bias && c < a.N) {                                      // N is a multiple of 8
      v.x += a.bias[c], v.y += a.bias[c + 1], v.z += a.bias[c + 2], v.w += a.bias[c + 3];
    }
    if (a.act)
      return make_float4(activate_on_store(v.x, a.act), activate_on_store(v.y, a.act), activate_on_store(v.z, a.act),
                         activate_on_store(v.w, a.act));
  }
  return v;
}
__device__ __forceinline__ uint2 panels_pack(const float4& v) { return make_uint2(pack2_bf16(v.x, v.y), pack2_bf16(v.z, v.w)); }

// ------------------------------------------------------------------------------- panels

template <int TM_, int TN_, int WM_, int WN_, int STAGES_>
struct Panels {
  static constexpr int TM = TM_, TN = TN_, WM = WM_, WN = WN_, STAGES = STAGES_, WAVES = WM * WN, PARTS = 1;
  static constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN, STAGE = (BM + BN) * 128, BYTES = STAGES * STAGE;
  static constexpr int LOADS = (BM + BN) / 8 / WAVES, READS = TM + TN, READS_A_GROUP = (READS + TN - 1) / TN;
  static_assert((BM + BN) / 8 % WAVES == 0, "every wave fills as many pieces of a stage");
  static_assert(BYTES <= 160 * 1024 && (STAGES - 1) * LOADS < 64, "shared memory; the count of loads on their way");
};

template <class T, int MODE>
__global__ void __launch_bounds__(64 * T::WAVES) gemm_panels_kernel(const PanelsArgs a) {
  constexpr int TM = T::TM, TN = T::TN, STAGES = T::STAGES, STAGE = T::STAGE, LOADS = T::LOADS;
  constexpr bool GATED = MODE == PANELS_GATED;
  extern __shared__ __attribute__((aligned(16))) unsigned char panel_stages[];
  const PanelsItem item = panels_item(a, T::BM, GATED ? T::BN / 2 : T::BN);
  if (!item.any) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const int wm = wave / T::WN, wn = wave - wm * T::WN;
  const int first = (int)((long long)item.slice * a.stages / a.slices);
  const int steps = (int)((long long)(item.slice + 1) * a.stages / a.slices) - first;      // at least one
  // piece p of a stage, 8 rows of it: rows of x, then of W; this wave fills pieces wave, wave + WAVES, ...
  unsigned off[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int row = 8 * (wave + T::WAVES * i) + (lane >> 3), k = 8 * ((lane & 7) ^ ((row >> 1) & 7));
    const int m = item.m0 + row < a.M ? item.m0 + row : a.M - 1;
    off[i] = 2u * (row < T::BM ? (unsigned)m * (unsigned)a.ldx + k
                               : (unsigned)panels_w_row<GATED, 8 * TN>(a, item.n0, row - T::BM) * (unsigned)a.ldw + k);
  }
  int until_end = steps - item.column % steps;
  const char* xb = reinterpret_cast<const char*>(a.x) + (size_t)(first + steps - until_end) * 128;
  const char* wb = reinterpret_cast<const char*>(a.w) + (size_t)(first + steps - until_end) * 128;
  auto next_stage = [&]() __attribute__((always_inline)) {
    const bool wrap = --until_end == 0;
    const int by = wrap ? 128 - 128 * steps : 128;
    xb += by, wb += by;
    if (wrap) until_end = steps;
  };
  const unsigned place = lds_place(panel_stages);
  auto load = [&](int i, unsigned to) __attribute__((always_inline)) {
    const int p = wave + T::WAVES * i;
    if (p < T::BM / 8) load16_to_lds_from(xb, off[i], place + to + p * 1024);
    else load16_to_lds_from_once(wb, off[i], place + to + p * 1024);
  };
  int at[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) at[s] = ((4 * s + g) ^ ((r >> 1) & 7)) << 4;
  const int xat = (16 * TM * wm + r) * 128, wat = (T::BM + 16 * TN * wn + r) * 128;
  tile_f32x4 acc[TN][TM];
#pragma unroll
  for (int n = 0; n < TN; ++n)
#pragma unroll
    for (int m = 0; m < TM; ++m) acc[n][m] = tile_f32x4{0.f, 0.f, 0.f, 0.f};
  TilePack x[2][TM], w[2][TN];
  // operand q of half s of a stage, those of the half's first products first
  auto operand = [&](const unsigned char* st, int s, int q) __attribute__((always_inline)) {
    if (q == 0) w[s][0].u4 = ld16(st + wat + at[s]);
    else if (q <= TM) x[s][q - 1].u4 = ld16(st + xat + at[s] + (q - 1) * 2048);
    else w[s][q - TM].u4 = ld16(st + wat + at[s] + (q - TM) * 2048);
  };
  auto operands = [&](const unsigned char* st, int s, int n) __attribute__((always_inline)) {
#pragma unroll
    for (int q = T::READS_A_GROUP * n; q < T::READS_A_GROUP * (n + 1); ++q)
      if (q < T::READS) operand(st, s, q);
  };
  auto products = [&](int s, int n) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < TM; ++m) acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[s][n].v, x[s][m].v, acc[n][m], 0, 0, 0);
  };
#pragma unroll
  for (int i = 0; i < STAGES; ++i)
    if (i < steps) {
#pragma unroll
      for (int j = 0; j < LOADS; ++j) load(j, i * STAGE);
      next_stage();
    }
  if (steps >= STAGES) loads_left<(STAGES - 1) * LOADS>();
  else loads_left<0>();
  bare_barrier();
#pragma unroll
  for (int q = 0; q < T::READS; ++q) operand(panel_stages, 0, q);
  int buf = 0;
  auto first_half = [&](const unsigned char* st) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      operands(st, 1, n);
      products(0, n);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // behind the wait and the barrier stage k + 1 is there and no wave still reads stage k, whose place the loads then take
  auto second_half = [&](auto loads) __attribute__((always_inline)) {
    const unsigned to = buf * STAGE;
    buf = buf == STAGES - 1 ? 0 : buf + 1;
    const unsigned char* const nx = panel_stages + buf * STAGE;
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      operands(nx, 0, n);
      if constexpr (decltype(loads)::value) {
#pragma unroll
        for (int j = n * LOADS / TN; j < (n + 1) * LOADS / TN; ++j) load(j, to);
      }
      products(1, n);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (decltype(loads)::value) next_stage();
  };
  int k = 0;
#pragma unroll 1
  for (; k + STAGES < steps; ++k) {
    first_half(panel_stages + buf * STAGE);
    loads_left<(STAGES - 2) * LOADS>();
    bare_barrier();
    second_half(std::integral_constant<bool, true>{});
  }
  // the last stages, all on their way: each waits for its successor alone
  auto last_stages = [&](auto self, auto left) __attribute__((always_inline)) -> void {
    constexpr int LEFT = decltype(left)::value;
    if constexpr (LEFT >= 2) {
      if (steps - k >= LEFT) {
        first_half(panel_stages + buf * STAGE);
        loads_left<(LEFT - 2) * LOADS>();
        bare_barrier();
        second_half(std::integral_constant<bool, false>{});
        ++k;
      }
      self(self, std::integral_constant<int, LEFT - 1>{});
    }
  };
  last_stages(last_stages, std::integral_constant<int, STAGES>{});
  first_half(panel_stages + buf * STAGE);
#pragma unroll
  for (int n = 0; n < TN; ++n) products(1, n);

  // acc[n][m]: lane (r, g) holds row 16 m + r of the wave's rows of x, columns 4 g .. 4 g + 3 of the n-th 16 of its rows of W
  constexpr int NT = GATED ? TN / 2 : TN;
  const int n_out = GATED ? a.N >> 1 : a.N, c0 = item.n0 + 16 * NT * wn;
  auto sums = [&](int n, int m) __attribute__((always_inline)) {
    return make_float4(acc[n][m][0], acc[n][m][1], acc[n][m][2], acc[n][m][3]);
  };
#pragma unroll
  for (int m = 0; m < TM; ++m) {
    const int row = item.m0 + 16 * (TM * wm + m) + r;
    if (row >= a.M) continue;
    if constexpr (MODE == PANELS_FLOAT) {
      float* const o = reinterpret_cast<float*>(a.out) + ((size_t)item.slice * a.M + row) * a.ldo;
#pragma unroll
      for (int n = 0; n < TN; ++n) {
        const int c = c0 + 16 * n + 4 * g;
        if (c < n_out) *reinterpret_cast<float4*>(o + c) = sums(n, m);
      }
    } else {
      bf16_t* const o = reinterpret_cast<bf16_t*>(a.out) + (size_t)row * a.ldo;
      uint2 v[NT];
#pragma unroll
      for (int n = 0; n < NT; ++n) v[n] = panels_pack(panels_finish<MODE>(a, sums(n, m), sums(GATED ? n + NT : n, m), c0 + 16 * n + 4 * g));
#pragma unroll
      for (int n = 0; n + 1 < NT; n += 2) {
        const uint4 both = pair_columns(v[n], v[n + 1]);
        const int c = c0 + 16 * n + pair_column(g);
        if (c < n_out) *reinterpret_cast<uint4*>(o + c) = both;
      }
      if constexpr (NT & 1) {
        const int c = c0 + 16 * (NT - 1) + 4 * g;
        if (c < n_out) *reinterpret_cast<uint2*>(o + c) = v[NT - 1];
      }
    }
  }
}

// ------------------------------------------------------------------------------- quarters

template <int TM_, int TN_>
struct Quarters {
  static constexpr int TM = TM_, TN = TN_, WAVES = 4, STAGES = 2, PARTS = WAVES;
  static constexpr int BM = 16 * TM, BN = 16 * TN, STAGE = (BM + BN) * 128, LOADS = (BM + BN) / 8, BYTES = WAVES * STAGES * STAGE;
  static_assert(BYTES <= 160 * 1024 && TM * TN * WAVES * 1024 <= BYTES, "shared memory; the waves' sums in the stages' place");
};

template <class T, int MODE>
__global__ void __launch_bounds__(64 * T::WAVES) gemm_quarters_kernel(const PanelsArgs a) {
  constexpr int TM = T::TM, TN = T::TN, STAGE = T::STAGE, LOADS = T::LOADS, XL = T::BM / 8;
  constexpr bool GATED = MODE == PANELS_GATED;
  constexpr int NT = GATED ? TN / 2 : TN;
  extern __shared__ __attribute__((aligned(16))) unsigned char panel_stages[];
  const PanelsItem item = panels_item(a, T::BM, 16 * NT);
  if (!item.any) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const int part = item.slice * T::WAVES + wave, parts = a.slices * T::WAVES;
  const int first = (int)((long long)part * a.stages / parts), steps = (int)((long long)(part + 1) * a.stages / parts) - first;   // at least one
  unsigned off[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int row = 8 * i + (lane >> 3), k = 8 * ((lane & 7) ^ ((row >> 1) & 7));
    const int m = item.m0 + row < a.M ? item.m0 + row : a.M - 1;
    off[i] = 2u * (i < XL ? (unsigned)m * (unsigned)a.ldx + k
                          : (unsigned)panels_w_row<GATED, 16 * NT>(a, item.n0, row - T::BM) * (unsigned)a.ldw + k);
  }
  int until_end = steps - item.column % steps;
  const char* xb = reinterpret_cast<const char*>(a.x) + (size_t)(first + steps - until_end) * 128;
  const char* wb = reinterpret_cast<const char*>(a.w) + (size_t)(first + steps - until_end) * 128;
  unsigned char* const mine = panel_stages + wave * 2 * STAGE;
  const unsigned place = lds_place(mine);
  auto fetch = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      if (i < XL) load16_to_lds_from(xb, off[i], place + buf * STAGE + i * 1024);
      else load16_to_lds_from_once(wb, off[i], place + buf * STAGE + i * 1024);
    }
    const bool wrap = --until_end == 0;
    const int by = wrap ? 128 - 128 * steps : 128;
    xb += by, wb += by;
    if (wrap) until_end = steps;
  };
  tile_f32x4 acc[TN][TM];
#pragma unroll
  for (int n = 0; n < TN; ++n)
#pragma unroll
    for (int m = 0; m < TM; ++m) acc[n][m] = tile_f32x4{0.f, 0.f, 0.f, 0.f};
  fetch(0);
  if (steps > 1) fetch(1);
  int buf = 0;
#pragma unroll 1
  for (int k = 0; k < steps; ++k) {
    if (k + 1 < steps) loads_left<LOADS>();              // those of the stage behind this one
    else loads_left<0>();
    const unsigned char* const st = mine + buf * STAGE;
    TilePack x[2][TM], w[2][TN];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int at = r * 128 + (((4 * s + g) ^ ((r >> 1) & 7)) << 4);
#pragma unroll
      for (int n = 0; n < TN; ++n) w[s][n].u4 = ld16(st + T::BM * 128 + n * 2048 + at);
#pragma unroll
      for (int m = 0; m < TM; ++m) x[s][m].u4 = ld16(st + m * 2048 + at);
    }
    auto products = [&](int s) __attribute__((always_inline)) {
#pragma unroll
      for (int n = 0; n < TN; ++n)
#pragma unroll
        for (int m = 0; m < TM; ++m) acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[s][n].v, x[s][m].v, acc[n][m], 0, 0, 0);
    };
    products(0);
    if (k + 2 < steps) {
      reads_done();
      fetch(buf);
    }
    buf ^= 1;
    products(1);
  }
  // the waves' sums, added in wave order: wave v finishes every fourth of the tile's 16 x 16 pieces
  __syncthreads();
  float4* const sums = reinterpret_cast<float4*>(panel_stages);
#pragma unroll
  for (int n = 0; n < TN; ++n)
#pragma unroll
    for (int m = 0; m < TM; ++m)
      sums[((n * TM + m) * T::WAVES + wave) * 64 + lane] = make_float4(acc[n][m][0], acc[n][m][1], acc[n][m][2], acc[n][m][3]);
  __syncthreads();
  auto total = [&](int n, int m) __attribute__((always_inline)) {
    const float4* const s = sums + (n * TM + m) * T::WAVES * 64 + lane;
    float4 t = s[0];
#pragma unroll
    for (int v = 1; v < T::WAVES; ++v) {
      const float4 u = s[64 * v];
      t.x += u.x, t.y += u.y, t.z += u.z, t.w += u.w;
    }
    return t;
  };
  const int n_out = GATED ? a.N >> 1 : a.N;
#pragma unroll
  for (int j = 0; j < (TM * NT + T::WAVES - 1) / T::WAVES; ++j) {
    const int u = j * T::WAVES + wave;
    if (u >= TM * NT) break;
    const int n = u % NT, m = u / NT, row = item.m0 + 16 * m + r, c = item.n0 + 16 * n + 4 * g;
    const float4 t = total(n, m);
    if (row >= a.M || c >= n_out) continue;
    if constexpr (MODE == PANELS_FLOAT)
      *reinterpret_cast<float4*>(reinterpret_cast<float*>(a.out) + ((size_t)item.slice * a.M + row) * a.ldo + c) = t;
    else
      *reinterpret_cast<uint2*>(reinterpret_cast<bf16_t*>(a.out) + (size_t)row * a.ldo + c) =
          panels_pack(panels_finish<MODE>(a, t, GATED ? total(n + NT, m) : t, c));
  }
}

// ------------------------------------------------------------------------------- launch

// The shapes, and what a block of each is estimated to take: `fixed` us around its K and `stage` us for every 64 values of it (of a
// quarter's, for the quarters), fitted to 6000 times of 8 matrices of 1024 to 24576 rows and 1024 to 12288 columns at 17 to 2048 rows.  The fastest of
// the shapes that were timed is missed by 1 % on average, 15 % at most; fewer than these cost more.
#define PANELS_SHAPES(PANEL, QUARTER)                                                                         \
  PANEL(2, 2, 1, 4, 6, 3.49f, 0.337f) PANEL(2, 2, 2, 2, 4, 3.36f, 0.265f) PANEL(2, 2, 2, 4, 6, 4.38f, 0.380f)  \
  PANEL(3, 2, 2, 2, 4, 3.75f, 0.318f) PANEL(3, 2, 2, 3, 6, 4.46f, 0.378f) PANEL(3, 4, 2, 2, 5, 5.10f, 0.438f)  \
  PANEL(4, 2, 2, 2, 6, 4.49f, 0.365f) PANEL(4, 2, 2, 4, 4, 5.67f, 0.497f) PANEL(5, 4, 2, 2, 4, 6.73f, 0.581f)  \
  PANEL(6, 2, 2, 4, 3, 6.70f, 0.597f) PANEL(4, 4, 4, 2, 3, 8.16f, 0.697f)                                      \
  QUARTER(2, 1, 1.88f, 0.377f) QUARTER(2, 2, 2.60f, 0.524f) QUARTER(3, 2, 2.87f, 0.621f) QUARTER(4, 2, 3.06f, 0.688f) \
  QUARTER(3, 4, 3.68f, 0.867f) QUARTER(4, 6, 4.52f, 1.359f)

struct PanelsShape {
  int rows, cols, parts, bytes;
  bool odd;                          // an odd number of 16-row pieces of W a wave: no gated unit
  float fixed, stage;
};
#define PANEL_ROW(TM, TN, WM, WN, ST, F, S) {16 * TM * WM, 16 * TN * WN, 1, (TM * WM + TN * WN) * 2048 * ST, TN % 2 != 0, F, S},
#define QUARTER_ROW(TM, TN, F, S) {16 * TM, 16 * TN, 4, (TM + TN) * 2048 * 8, TN % 2 != 0, F, S},
static const PanelsShape panels_shapes[] = {PANELS_SHAPES(PANEL_ROW, QUARTER_ROW)};
static const int panels_shape_count = sizeof(panels_shapes) / sizeof(panels_shapes[0]);

extern "C" int ullm_gemm_panels_shapes(void) { return panels_shape_count; }

static long long panels_blocks(const PanelsShape& s, int M, int N, int mode, int slices) {
  const int n_out = mode == PANELS_GATED ? N / 2 : N, cols = mode == PANELS_GATED ? s.cols / 2 : s.cols;
  return (long long)((M + s.rows - 1) / s.rows) * ((n_out + cols - 1) / cols) * slices;
}

// Blocks of a product by a shape (and slices) that takes it.
extern "C" int ullm_gemm_panels_blocks(int M, int N, int mode, int shape, int slices) {
  if (shape < 0 || shape >= panels_shape_count) return 0;
  const long long blocks = panels_blocks(panels_shapes[shape], M, N, mode, slices);
  return blocks < (1LL << 24) ? (int)blocks : 1 << 24;
}

// Whether a shape and a number of slices take the product: K in whole stages, one at least for every part of it; rows whose ends
// 32-bit byte offsets reach.
extern "C" int ullm_gemm_panels_supports(int M, int N, int K, int ldx, int ldw, int mode, int shape, int slices) {
  if (M < 1 || N < 8 || K < 64 || K % 64 || mode < PANELS_STORE || mode > PANELS_FLOAT || shape < 0 || shape >= panels_shape_count)
    return 0;
  const PanelsShape& s = panels_shapes[shape];
  return N % (mode == PANELS_GATED ? 16 : 8) == 0 && !(mode == PANELS_GATED && s.odd) && slices >= 1 && (slices == 1 || mode == PANELS_FLOAT) &&
         K / 64 >= slices * s.parts && ldx % 8 == 0 && ldw % 8 == 0 && ldx >= K && ldw >= K && (long long)M * ldx < (1LL << 31) &&
         (long long)N * ldw < (1LL << 31) && panels_blocks(s, M, N, mode, slices) < (1LL << 24);
}

// The shape and slices (at most max_slices) estimated to be the fastest: shape | slices << 8 | (more than one round of blocks) << 16
// | its time in eighths of a us (8191 at most) << 17, or -1 where none takes the product.  A block's time, and the time its bytes take at 5.6 TB/s, count as the cube root of the sum
// of their cubes: what is bound by neither alone takes longer than either.  A shape of at most half a unit's shared memory runs two blocks a unit side by
// side in twice the time of one.  Slices cost their consumer's reading of them.
extern "C" int ullm_gemm_panels_plan(int M, int N, int K, int mode, int max_slices) {
  static const int tried[] = {1, 2, 3, 4, 6, 8};
  int best = -1;
  float least = 0.f;
  for (int i = 0; i < panels_shape_count; ++i) {
    const PanelsShape& s = panels_shapes[i];
    for (int slices : tried) {
      if (slices > max_slices || !ullm_gemm_panels_supports(M, N, K, K, K, mode, i, slices)) continue;
      const long long blocks = panels_blocks(s, M, N, mode, slices);
      const float rounds = 2 * s.bytes > 160 * 1024 ? (float)((blocks + 255) / 256) : blocks <= 256 ? 1.f : 0.5f * (float)((blocks + 127) / 128);
      const float outs = (float)M * N * (mode == PANELS_FLOAT ? 4e-6f * slices : mode == PANELS_GATED ? 1e-6f : 2e-6f);      // MB
      const float bytes = 2e-6f * K * ((float)N + (float)M) + outs;
      const float work = rounds * (s.fixed + s.stage * (float)K / (64.f * slices * s.parts)), memory = bytes / 5.6f;
      const float us = cbrtf(work * work * work + memory * memory * memory) + (mode == PANELS_FLOAT ? outs / 8.f : 0.f);
      if (best < 0 || us < least) best = i | slices << 8 | (rounds > 1.f ? 1 << 16 : 0), least = us;
    }
  }
  return best < 0 ? best : best | (least < 1023.f ? (int)(8.f * least) : 8191) << 17;
}

template <class T, int MODE, class Kernel>
static int launch_panels(Kernel kernel, const PanelsArgs& a, long long blocks, hipStream_t stream) {
  static const hipError_t allowed = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, T::BYTES);
  if (allowed != hipSuccess) return (int)allowed;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(8 * ((blocks + 7) / 8))), dim3(64 * T::WAVES), T::BYTES, stream, a);
  ULLM_LAUNCH_CHECK();
}

// x bfloat16 [M, K], row stride ldx; W bfloat16 [N, K], row stride ldw; out [M, ldo] bfloat16, or float32 [slices, M, ldo].  bias
// float32 [N] or null, act an activation (kind + 1, 0: none; store only); limit, alpha the gated unit's.
extern "C" int ullm_gemm_panels(const void* x, int ldx, const void* w, int ldw, const float* bias, void* out, int ldo, int M, int N,
                                int K, int mode, int shape, int slices, float limit, float alpha, int act, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (!ullm_gemm_panels_supports(M, N, K, ldx, ldw, mode, shape, slices)) return ULLM_ERR_SHAPE;
  if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15 || ldo % 8 || ldo < (mode == PANELS_GATED ? N / 2 : N)) return ULLM_ERR_SHAPE;
  if ((bias || act) && mode != PANELS_STORE) return ULLM_ERR_UNSUPPORTED;
  if (act < 0 || act > 3 || (limit > 0.f && mode != PANELS_GATED)) return ULLM_ERR_UNSUPPORTED;
  const PanelsShape& s = panels_shapes[shape];
  const int cols = mode == PANELS_GATED ? s.cols / 2 : s.cols, n_out = mode == PANELS_GATED ? N / 2 : N;
  const PanelsArgs a{(const bf16_t*)x, ldx, (const bf16_t*)w, ldw, bias, out, ldo, M, N, K / 64, slices, (M + s.rows - 1) / s.rows,
                     (n_out + cols - 1) / cols, limit, alpha, act};
  const long long blocks = panels_blocks(s, M, N, mode, slices);
  int i = 0;
#define MODES(T, KERNEL)                                                                                             \
  if (mode == PANELS_STORE) return launch_panels<T, PANELS_STORE>(KERNEL<T, PANELS_STORE>, a, blocks, stream);       \
  if (mode == PANELS_FLOAT) return launch_panels<T, PANELS_FLOAT>(KERNEL<T, PANELS_FLOAT>, a, blocks, stream);       \
  if constexpr (T::TN % 2 == 0) return launch_panels<T, PANELS_GATED>(KERNEL<T, PANELS_GATED>, a, blocks, stream);
#define PANEL_GO(TM, TN, WM, WN, ST, F, S)    \
  if (shape == i++) {                         \
    using T = Panels<TM, TN, WM, WN, ST>;     \
    MODES(T, gemm_panels_kernel)              \
  }
#define QUARTER_GO(TM, TN, F, S)     \
  if (shape == i++) {                \
    using T = Quarters<TM, TN>;      \
    MODES(T, gemm_quarters_kernel)   \
  }
  PANELS_SHAPES(PANEL_GO, QUARTER_GO)
  return ULLM_ERR_SHAPE;
}
