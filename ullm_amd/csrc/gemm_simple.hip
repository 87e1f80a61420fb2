// C[M, N] = A[M, K] * W[N, K]^T (+ bias[N]) with 32-bit products and sums in a fixed K order, on the 32-bit matrix
// instruction v_mfma_f32_16x16x4_f32 (whose products and sums are full 32-bit: no rounding of the inputs).
// The product of row m never depends on M, on the other rows or on the tile it lies in: every variant below adds the products
// in the order of K into one chain of sums per output (mfma_f32.h), so a token's result is the same in every batch, and the
// bits are those of a plain loop of fma over K.  This is the matrix product of the float32
// mode and the general fallback for bfloat16 operands (widened exactly on their way to shared memory).
// Weights are [out, in] as the reference stores them for F.linear (ullm/layers/linear.py:165,268).
//
// What bounds it: the matrix pipe (157 TFLOP/s in 32-bit) where the tiles fill the chip, the chain over K where they do
// not (a 16 x 16 tile adds 4 k in 32 cycles).  Hence the tile sizes: large ones read shared memory and the second-level
// cache less per product, small ones make more blocks.  A unit that has one block has one wave a SIMD: whatever is not
// put between the products of that wave is time the pipe stands still.  So the next stage is written, and the one after the next
// two fetched, piece by piece between the products, operands are read a chunk ahead, and the only wait a stage is its barrier.
// In stages that were written in one go behind their products, with a condition on fetched values that waited for all of them:
// 500 rows, 4096 outputs, K = 1024 43 -> 39 us (109 TFLOP/s), 6144 outputs 60 -> 56, 1024 outputs and K = 2048 34 -> 24, K = 3072
// 49 -> 36; 40 rows 23 -> 16 and 33 -> 23; 2048 rows of 4096 outputs 156 -> 142.  Stages that are exchanged between lanes in
// registers and written 16 bytes at a time, from rows read in half lines, are slower (43 us for 36, 56 for 44).
#include "mfma_f32.h"

#include <algorithm>

// A block of four waves takes BM rows of A against BN rows of W, WGM waves side by side along M.  A stage is BK values of
// K: rows in shared memory whose 16-byte piece c of row r lies at piece c ^ ((r >> 1) & 7) (the 16 lanes the hardware
// serves together then read different bank groups); two stages take turns, and a stage is fetched into registers three
// stages before its products.  A barrier costs the smaller tiles the more, so they
// take 64 values a stage.  Lane (r, g) of a wave reads k = g, 4 + g, 8 + g, 12 + g of its row's chunk at
// once (they are written side by side) and holds out[row r of A][columns 4g .. 4g + 3] of each 16 x 16 tile.  VEC: four values a load (K and the row lengths are
// multiples of four values and the addresses of that alignment), 2 where also K is whole stages; 0: one by one.  No load stands under a condition: a
// row past the end reads the last row, a piece past K the row's last piece (replaced by zeros); neither is stored.
template <typename TA, typename TW, typename TC, int BM, int BN, int WGM, int BK, int VEC, bool GATED = false>
__global__ void __launch_bounds__(256)
gemm_simple_kernel(const TA* __restrict__ A, int lda, const TW* __restrict__ W, int ldw, const float* __restrict__ bias,
                   TC* __restrict__ C, int ldc, int M, int N, int K, int m_tiles, int n_tiles) {
  constexpr int WGN = 4 / WGM, TM = BM / 16 / WGM, TN = BN / 16 / WGN, PR = BK / 4, STEP = 256 / PR, CHUNKS = BK / 16;
  static_assert(CHUNKS % 2 == 0, "a stage's first chunk lies in the same registers every time");
  constexpr int AP = (BM + STEP - 1) / STEP, WP = (BN + STEP - 1) / STEP;  // pieces a thread fetches a stage
  __shared__ __attribute__((aligned(16))) unsigned char stages[2][(BM + BN) * BK * 4];
  // die d (blocks go to the 8 dies round-robin) takes the d-th eighth of the tiles, all rows of A for a strip of W before
  // the next strip: what a die's second-level cache holds of W serves all of its row tiles
  const int total = m_tiles * n_tiles, per_die = (total + 7) / 8;
  const int item = ((int)blockIdx.x & 7) * per_die + ((int)blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_die || item >= total) return;
  const int m0 = item % m_tiles * BM, n0 = item / m_tiles * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, g = lane >> 4;
  const int wm = wave % WGM * TM * 16, wn = wave / WGM * TN * 16;
  const int pc = tid % PR, prow = tid / PR;
  const TA* asrc[AP];
  const TW* wsrc[WP];
  int aput[AP], wput[WP], alow[AP], wlow[WP];
#pragma unroll
  for (int i = 0; i < AP; ++i) {
    const int row = (prow + STEP * i) % BM;              // more threads than pieces: two fetch and write the same
    asrc[i] = A + (size_t)(m0 + row < M ? m0 + row : M - 1) * lda;
    aput[i] = row * BK * 4 + (((pc & ~3) ^ ((row >> 1) & 4)) << 4) + 4 * (pc & 3), alow[i] = (row >> 1) & 3;
  }
#pragma unroll
  for (int i = 0; i < WP; ++i) {
    const int row = (prow + STEP * i) % BN;
    int of = n0 + row < N ? n0 + row : N - 1;
    if constexpr (GATED) {                               // 16 rows of gate, then the same 16 of up
      const int column = n0 / 2 + (row >> 5) * 16 + (row & 15), I = N / 2;
      of = ((row >> 4) & 1) * I + (column < I ? column : I - 1);
    }
    wsrc[i] = W + (size_t)of * ldw;
    wput[i] = (BM + row) * BK * 4 + (((pc & ~3) ^ ((row >> 1) & 4)) << 4) + 4 * (pc & 3), wlow[i] = (row >> 1) & 3;
  }
  // piece p of a stage (those of A first) on its way to registers
  float4 reg[2][AP + WP];
  auto fetch = [&](int set, int p, int k0) __attribute__((always_inline)) {
    const int k = k0 + 4 * pc;
    if (VEC) {
      const int kk = k < K ? k : K - 4;
      if (p < AP) reg[set][p] = ld4_f32(asrc[p] + kk);
      else reg[set][p] = ld4_f32(wsrc[p - AP] + kk);
    } else {
      auto one = [&](auto src) __attribute__((always_inline)) {
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = ld_f32(src + (k + j < K ? k + j : K - 1));
        return make_float4(v[0], v[1], v[2], v[3]);
      };
      if (p < AP) reg[set][p] = one(asrc[p]);
      else reg[set][p] = one(wsrc[p - AP]);
    }
  };
  // value e of a piece goes to the chunk's piece e: a lane group's 16 bytes are then values g, 4 + g, 8 + g, 12 + g of the chunk
  // (64 lanes write one value each to 64 different banks).  Zeros are put in here: a condition on a fetched value any earlier
  // would wait for the fetch (33 rows of 2048 outputs, K = 3001, whose values come one by one, 71 us, 46 so).
  auto put = [&](int set, int p, int buf, int k0) __attribute__((always_inline)) {
    float v[4] = {reg[set][p].x, reg[set][p].y, reg[set][p].z, reg[set][p].w};
    if (VEC < 2) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = k0 + 4 * pc + (VEC ? 0 : e) < K ? v[e] : 0.f;
    }
    unsigned char* row = stages[buf] + (p < AP ? aput[p] : wput[p - AP]);
    const int low = p < AP ? alow[p] : wlow[p - AP];
#pragma unroll
    for (int e = 0; e < 4; ++e) *reinterpret_cast<float*>(row + ((e ^ low) << 4)) = v[e];
  };
  f32x4_t acc[TN][TM];
#pragma unroll
  for (int n = 0; n < TN; ++n)
#pragma unroll
    for (int m = 0; m < TM; ++m) acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  f32x4_t a[2][TM], w[2][TN];
  auto take = [&](int set, int buf, int c) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < TM; ++m) {
      const int row = wm + 16 * m + r;
      a[set][m] = *reinterpret_cast<const f32x4_t*>(stages[buf] + row * BK * 4 + (((4 * c + g) ^ ((row >> 1) & 7)) << 4));
    }
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      const int row = wn + 16 * n + r;
      w[set][n] = *reinterpret_cast<const f32x4_t*>(stages[buf] + (BM + row) * BK * 4 + (((4 * c + g) ^ ((row >> 1) & 7)) << 4));
    }
  };
  // Stage k0 from its buffer, its first chunk taken already; `set` holds the next stage, the other set the one after it, both on
  // their way.  A chunk is taken while the one before it is multiplied, over the barrier too: that stands ahead of the last
  // chunk's products, when the last chunk has been taken (this buffer is free) and the next stage is written.  Between the
  // products of the chunks before it the next stage is written, each piece's registers being fetched anew behind it.
  auto stage = [&](int buf, int set, int k0) __attribute__((always_inline)) {
    constexpr int P = AP + WP, SLOTS = 4 * (CHUNKS - 1);
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
      const bool last = c == CHUNKS - 1;
      if (last) __syncthreads();
      take((c + 1) & 1, last ? buf ^ 1 : buf, last ? 0 : c + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int n = 0; n < TN; ++n)
#pragma unroll
          for (int m = 0; m < TM; ++m)
            acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[c & 1][n][i], a[c & 1][m][i], acc[n][m], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = 0; p < P; ++p)
          if (!last && p * SLOTS / P == 4 * c + i) {
            put(set, p, buf ^ 1, k0 + BK);
            fetch(set, p, k0 + 3 * BK);
          }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
#pragma unroll
  for (int s = 0; s < 2; ++s)
#pragma unroll
    for (int p = 0; p < AP + WP; ++p) fetch(s, p, s * BK);
#pragma unroll
  for (int p = 0; p < AP + WP; ++p) {
    put(0, p, 0, 0);
    fetch(0, p, 2 * BK);
  }
  __syncthreads();
  take(0, 0, 0);
  for (int k0 = 0;; k0 += 2 * BK) {
    stage(0, 1, k0);
    if (k0 + BK >= K) break;
    stage(1, 0, k0 + BK);
    if (k0 + 2 * BK >= K) break;
  }
  if constexpr (GATED) {
    static_assert(TN == 2 && sizeof(TC) == 4, "a wave holds gate and up of the same columns");
#pragma unroll
    for (int m = 0; m < TM; ++m) {
      const int gm = m0 + wm + 16 * m + r, column = (n0 + wn) / 2 + 4 * g, I = N / 2;
      if (gm >= M) continue;
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = acc[0][m][i] / (1.f + expf(-acc[0][m][i])) * acc[1][m][i];
      TC* o = C + (size_t)gm * ldc + column;
      if (column + 3 < I && (ldc & 3) == 0 && !((uintptr_t)C & 15)) {
        *reinterpret_cast<float4*>(o) = make_float4(v[0], v[1], v[2], v[3]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (column + i < I) st_f32(o + i, v[i]);
      }
    }
    return;
  }
#pragma unroll
  for (int m = 0; m < TM; ++m) {
    const int gm = m0 + wm + 16 * m + r;
    if (gm >= M) continue;
#pragma unroll
    for (int n = 0; n < TN; ++n) {
      const int gn = n0 + wn + 16 * n + 4 * g;
      TC* o = C + (size_t)gm * ldc + gn;
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        v[i] = acc[n][m][i];
        if (bias) v[i] += bias[gn + i < N ? gn + i : N - 1];
      }
      if (sizeof(TC) == 4 && gn + 3 < N && (ldc & 3) == 0 && !((uintptr_t)C & 15)) {
        *reinterpret_cast<float4*>(o) = make_float4(v[0], v[1], v[2], v[3]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (gn + i < N) st_f32(o + i, v[i]);
      }
    }
  }
}

// Compute units of the current device (asked once per device).
static int simple_compute_units() {
  static int units[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (units[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    units[dev] = n;
  }
  return units[dev];
}

// How many tiles the fullest unit takes.
static long long fullest(long long M, long long N, int bm, int bn, int units) {
  return (((M + bm - 1) / bm) * ((N + bn - 1) / bn) + units - 1) / units;
}

// How long each tile takes at K = 1024, in us: what begins and ends a launch and, for every tile that the fullest compute
// unit takes, its products (blocks side by side on a unit share the matrix pipe).  Fitted to 15 numbers of rows by 12
// matrices, where the choice is within 5 % of the fastest tile; the constants grow alike with K.  Small tiles win while
// every unit has one at most (K = 3072, 250 rows of 1024 outputs: 25 us, 35 in tiles of 64 x 32, 57 of 64 x 64), 64 x 64 when
// units have many (500 rows of 4096: 50, 40, 39 us), stages of 32 values for 64 x 32 from two on; one to sixteen rows
// of many outputs are bound by the matrix's bytes (151 936: 110 us, 122 in tiles of 32 x 32).
static int product_tile(int M, int N, int units) {
  auto time = [&](int bm, int bn, double once, double each) { return once + each * (double)fullest(M, N, bm, bn, units); };
  const double times[] = {time(32, 32, 5.0, 5.6), time(32, 64, 4.0, 9.9), time(64, 32, 4.0, 9.9), time(64, 32, 6.5, 9.0),
                          time(64, 64, 4.0, 17.2), M <= 16 ? time(16, 64, 6.0, 5.0) : 1e30};
  return (int)(std::min_element(times, times + 6) - times);
}

template <typename TA, typename TW, typename TC, int VEC>
static void launch(const void* A, int lda, const void* W, int ldw, const float* bias, void* C, int ldc, int M, int N, int K,
                   hipStream_t stream) {
#define TILE(BM, BN, WGM, BK) do { \
    const int mt = (M + BM - 1) / BM, nt = (N + BN - 1) / BN; \
    hipLaunchKernelGGL((gemm_simple_kernel<TA, TW, TC, BM, BN, WGM, BK, VEC>), dim3(8 * (((unsigned)mt * nt + 7) / 8)), dim3(256), 0, \
                       stream, (const TA*)A, lda, (const TW*)W, ldw, bias, (TC*)C, ldc, M, N, K, mt, nt); } while (0)
  // operands one by one: what is fetched counts, so large tiles where they give a unit one and a half (400 rows of 5000 outputs, K = 770: 75 us, 92 in tiles of
  // 32 x 32)
  const int units = simple_compute_units();
  const bool large = VEC == 0 && ((M + 63) / 64) * ((N + 63LL) / 64) * 2 >= 3 * units;
  switch (large ? 4 : product_tile(M, N, units)) {
    case 0: TILE(32, 32, 2, 64); break;
    case 1: TILE(32, 64, 2, 64); break;
    case 2: TILE(64, 32, 2, 64); break;
    case 3: TILE(64, 32, 2, 32); break;
    case 4: TILE(64, 64, 2, 32); break;
    default: TILE(16, 64, 1, 64);
  }
#undef TILE
}

extern "C" int ullm_gemm_simple(const void* A, int lda, const void* W, int ldw, const float* bias,
                                void* C, int ldc, int M, int N, int K, int a_dtype, int w_dtype,
                                int c_dtype, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || lda < K || ldw < K || ldc < N) return ULLM_ERR_SHAPE;
  if ((a_dtype | w_dtype | c_dtype) & ~1) return ULLM_ERR_DTYPE;
  if (((long long)M + 15) / 16 * (((long long)N + 31) / 32) > 0x3fffffffLL) return ULLM_ERR_SHAPE;
  const bool vec = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && !((uintptr_t)A & (a_dtype == ULLM_F32 ? 15 : 7)) &&
                   !((uintptr_t)W & (w_dtype == ULLM_F32 ? 15 : 7));
#define GO(TA, TW, TC) do { \
    if (vec && K % 64 == 0) launch<TA, TW, TC, 2>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream); \
    else if (vec) launch<TA, TW, TC, 1>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream); \
    else launch<TA, TW, TC, 0>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream); } while (0)
  const int key = a_dtype * 4 + w_dtype * 2 + c_dtype;
  switch (key) {
    case 0: GO(float, float, float); break;
    case 7: GO(bf16_t, bf16_t, bf16_t); break;
    case 6: GO(bf16_t, bf16_t, float); break;
    case 2: GO(float, bf16_t, float); break;
    case 4: GO(bf16_t, float, float); break;     // 32-bit weights on rounded activations (a router)
    default: return ULLM_ERR_DTYPE;
  }
#undef GO
  ULLM_LAUNCH_CHECK();
}

// Whether the gated product takes tiles of 32 rows, not of 64: us a tile of the fullest unit, as in product_tile.
static bool gated_in_small_tiles(int M, int I, int units) {
  return 9.9 * fullest(M, 2LL * I, 32, 64, units) <= 17.2 * fullest(M, 2LL * I, 64, 64, units);
}

// 1 where ullm_gemm_simple_gated is expected ahead of the product and the activation kernel behind it, on a device of `units` compute units.  It has
// two tiles, those in which a wave holds pairs of gate and up; the product takes smaller or longer ones where these fill the chip better, most of
// all where tiles of 32 x 32 are one a unit at most: 64 rows of 2 x 1408 columns, K = 2048, 19.7 us in two kernels and 24.6 in one, 17 of 2 x 3072,
// K = 1024, 13.4 and 14.5, 192 of 2 x 5504, K = 2048, 95.0 and 98.7; but 65 of the first 27.6 and 24.7, 500 of the second 59.9 and 54.3.
// Times in us of each tile, once and for every one that the fullest unit takes at K = 1024, and of the activation, by 390 pairs (17 to 2048
// rows, 13 matrices): the choice is within 1.5 % of the better one in all; a tie is the gated product's.
// Not `captured` (for a graph's replays): the host launches one after the other, and two launches take it 16 us (17 rows of 2 x 512 columns, K = 512: 8.3 and
// 8.8 us in a graph, 15.2 and 8.3 without; prompts of 17 tokens of a 0.6B model 2.88 and 2.81 ms, decode of 17 requests the other way round).
extern "C" int ullm_gemm_simple_gated_ahead(int M, int I, int K, int captured, int units) {
  if (M <= 16 || I <= 0 || K <= 0 || units <= 0 || I > 0x3fffffff) return 0;
  auto time = [&](int bm, int bn, double once, double each) { return once + each * K / 1024.0 * (double)fullest(M, 2LL * I, bm, bn, units); };
  double two = 2.04 + 1.82e-6 * M * I;                     // the activation kernel
  switch (product_tile(M, 2 * I, units)) {
    case 0: two += time(32, 32, 3.67, 6.36); break;
    case 1: two += time(32, 64, 4.6, 10.17); break;
    case 2: two += time(64, 32, 4.6, 10.17); break;
    case 3: two += time(64, 32, 3.47, 9.47); break;
    default: two += time(64, 64, 6.0, 16.85);
  }
  if (!captured && two < 16.0) two = 16.0;
  const double one = gated_in_small_tiles(M, I, units) ? time(32, 64, 4.06, 10.14) : time(64, 64, 5.63, 16.8);
  return one <= 1.005 * two;
}

// silu(A G^T) * (A U^T) of 32-bit operands, W = G | U [2 I, K], out [M, I]: the product above with the gated unit on store, in the tiles in which a
// wave holds gate and up of the same columns.  The bits are those of the product and the activation kernel behind it.  us for
// both and for this one, 2 x 3072 columns, K = 1024: 40 rows 16.9, 14.3, 130 27.3, 23.9, 500 59.9, 54.3, 2048 227, 211; 2 x 6144, K = 2048: 40 rows 43, 40,
// 100 64.0, 66.6 (64 x 32 is ahead there, which has no pairs), 1000 422, 407.
extern "C" int ullm_gemm_simple_gated(const float* A, int lda, const float* W, int ldw, float* out, int ldo, int M, int I, int K,
                                      hipStream_t stream) {
  if (M <= 0 || I <= 0) return 0;
  if (K <= 0 || lda < K || ldw < K || ldo < I || I > 0x3fffffff) return ULLM_ERR_SHAPE;
  if (((long long)M + 31) / 32 * (((long long)I + 31) / 32) > 0x3fffffffLL) return ULLM_ERR_SHAPE;
  const bool vec = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && !(((uintptr_t)A | (uintptr_t)W) & 15);
  const int N = 2 * I, nt = (I + 31) / 32;
#define TILE(BM, BK, VEC) do { \
    const int mt = (M + BM - 1) / BM; \
    hipLaunchKernelGGL((gemm_simple_kernel<float, float, float, BM, 64, 2, BK, VEC, true>), dim3(8 * (((unsigned)mt * nt + 7) / 8)), dim3(256), \
                       0, stream, A, lda, W, ldw, (const float*)nullptr, out, ldo, M, N, K, mt, nt); } while (0)
#define GO(VEC) do { if (small) TILE(32, 64, VEC); else TILE(64, 32, VEC); } while (0)
  const bool small = gated_in_small_tiles(M, I, simple_compute_units());
  if (vec && K % 64 == 0) GO(2);
  else if (vec) GO(1);
  else GO(0);
#undef GO
#undef TILE
  ULLM_LAUNCH_CHECK();
}
