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
// cache less per product, small ones make more blocks.  Against a 64 x 64 tile of scalar multiply-adds whose operands came
// one value a load: 500 rows, 4096 outputs, K = 1024 122 -> 49 us (85 TFLOP/s), 1024 outputs, K = 3072 407 -> 52 us; 2048
// rows, 4096 outputs 272 -> 179 us; one row of 151 936 outputs 434 -> 115 us (5.4 TB/s).
#include "mfma_f32.h"

// A block of four waves takes BM rows of A against BN rows of W, WGM waves side by side along M.  A stage is BK values of
// K: rows in shared memory whose 16-byte piece c of row r lies at piece c ^ ((r >> 1) & 7) (the 16 lanes the hardware
// serves together then read different bank groups); two stages take turns, and a stage is fetched into registers two
// stages before its products.  A stage costs about 600 cycles of writing, barrier and reading beside its products, so the
// smaller tiles take 64 values a stage.  Lane (r, g) of a wave reads k = g, 4 + g, 8 + g, 12 + g of its row's chunk at
// once (they are written side by side) and holds out[row r of A][columns 4g .. 4g + 3] of each 16 x 16 tile.  VEC: four values a load (K and the row lengths are
// multiples of four values and the addresses of that alignment); else one by one.  No load stands under a condition: a
// row past the end reads the last row, a piece past K the row's last piece (replaced by zeros); neither is stored.
template <typename TA, typename TW, typename TC, int BM, int BN, int WGM, int BK, bool VEC>
__global__ void __launch_bounds__(256)
gemm_simple_kernel(const TA* __restrict__ A, int lda, const TW* __restrict__ W, int ldw, const float* __restrict__ bias,
                   TC* __restrict__ C, int ldc, int M, int N, int K, int m_tiles, int n_tiles) {
  constexpr int WGN = 4 / WGM, TM = BM / 16 / WGM, TN = BN / 16 / WGN, PR = BK / 4, STEP = 256 / PR;
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
    wsrc[i] = W + (size_t)(n0 + row < N ? n0 + row : N - 1) * ldw;
    wput[i] = (BM + row) * BK * 4 + (((pc & ~3) ^ ((row >> 1) & 4)) << 4) + 4 * (pc & 3), wlow[i] = (row >> 1) & 3;
  }
  float4 areg[2][AP], wreg[2][WP];
  auto fetch = [&](int set, int k0) __attribute__((always_inline)) {
    const int k = k0 + 4 * pc;
    if (VEC) {
      const bool in = k < K;
      const int kk = in ? k : K - 4;
#pragma unroll
      for (int i = 0; i < AP; ++i) areg[set][i] = ld4_f32(asrc[i] + kk);
#pragma unroll
      for (int i = 0; i < WP; ++i) wreg[set][i] = ld4_f32(wsrc[i] + kk);
      if (!in) {
#pragma unroll
        for (int i = 0; i < AP; ++i) areg[set][i] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int i = 0; i < WP; ++i) wreg[set][i] = make_float4(0.f, 0.f, 0.f, 0.f);
      }
    } else {
      auto one = [&](auto* src) __attribute__((always_inline)) {
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float x = ld_f32(src + (k + j < K ? k + j : K - 1));
          v[j] = k + j < K ? x : 0.f;
        }
        return make_float4(v[0], v[1], v[2], v[3]);
      };
#pragma unroll
      for (int i = 0; i < AP; ++i) areg[set][i] = one(asrc[i]);
#pragma unroll
      for (int i = 0; i < WP; ++i) wreg[set][i] = one(wsrc[i]);
    }
  };
  // value e of a piece goes to the chunk's piece e: a lane group's 16 bytes are then values g, 4 + g, 8 + g, 12 + g of the chunk
  // (64 lanes write one value each to 64 different banks)
  auto put = [&](int set, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < AP; ++i) {
      const float v[4] = {areg[set][i].x, areg[set][i].y, areg[set][i].z, areg[set][i].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) *reinterpret_cast<float*>(stages[buf] + aput[i] + ((e ^ alow[i]) << 4)) = v[e];
    }
#pragma unroll
    for (int i = 0; i < WP; ++i) {
      const float v[4] = {wreg[set][i].x, wreg[set][i].y, wreg[set][i].z, wreg[set][i].w};
#pragma unroll
      for (int e = 0; e < 4; ++e) *reinterpret_cast<float*>(stages[buf] + wput[i] + ((e ^ wlow[i]) << 4)) = v[e];
    }
  };
  f32x4_t acc[TN][TM];
#pragma unroll
  for (int n = 0; n < TN; ++n)
#pragma unroll
    for (int m = 0; m < TM; ++m) acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto products = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < BK / 16; ++c) {
      f32x4_t a[TM], w[TN];
#pragma unroll
      for (int m = 0; m < TM; ++m) {
        const int row = wm + 16 * m + r;
        a[m] = *reinterpret_cast<const f32x4_t*>(stages[buf] + row * BK * 4 + (((4 * c + g) ^ ((row >> 1) & 7)) << 4));
      }
#pragma unroll
      for (int n = 0; n < TN; ++n) {
        const int row = wn + 16 * n + r;
        w[n] = *reinterpret_cast<const f32x4_t*>(stages[buf] + (BM + row) * BK * 4 + (((4 * c + g) ^ ((row >> 1) & 7)) << 4));
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int n = 0; n < TN; ++n)
#pragma unroll
          for (int m = 0; m < TM; ++m) acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[n][i], a[m][i], acc[n][m], 0, 0, 0);
    }
  };
  fetch(0, 0);
  put(0, 0);
  __syncthreads();
  fetch(0, BK);
  for (int k0 = 0; k0 < K; k0 += 2 * BK) {
    // stage k0 lies in buffer 0, set 0 holds stage k0 + BK (on its way)
    fetch(1, k0 + 2 * BK);
    products(0);
    if (k0 + BK < K) put(0, 1);
    __syncthreads();
    if (k0 + BK >= K) break;
    fetch(0, k0 + 3 * BK);
    products(1);
    if (k0 + 2 * BK < K) put(1, 0);
    __syncthreads();
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

template <typename TA, typename TW, typename TC, bool VEC>
static void launch(const void* A, int lda, const void* W, int ldw, const float* bias, void* C, int ldc, int M, int N, int K,
                   hipStream_t stream) {
#define TILE(BM, BN, WGM, BK) do { \
    const int mt = (M + BM - 1) / BM, nt = (N + BN - 1) / BN; \
    hipLaunchKernelGGL((gemm_simple_kernel<TA, TW, TC, BM, BN, WGM, BK, VEC>), dim3(8 * (((unsigned)mt * nt + 7) / 8)), dim3(256), 0, \
                       stream, (const TA*)A, lda, (const TW*)W, ldw, bias, (TC*)C, ldc, M, N, K, mt, nt); } while (0)
  // 64 x 64 from where they give every compute unit a block and a half: 500 rows x 4096 outputs (512 tiles) 48 us against 64 in
  // tiles of 32, 500 x 1024 (128 tiles) the other way round
  auto tiles = [&](long long bm, long long bn) { return ((M + bm - 1) / bm) * ((N + bn - 1) / bn); };
  if (M <= 16) TILE(16, 64, 1, 64);
  else if (tiles(64, 64) >= 400) TILE(64, 64, 2, 32);
  else TILE(32, 32, 2, 64);
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
    if (vec) launch<TA, TW, TC, true>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream); \
    else launch<TA, TW, TC, false>(A, lda, W, ldw, bias, C, ldc, M, N, K, stream); } while (0)
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
