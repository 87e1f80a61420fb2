// Large bfloat16 products out = x W^T on the matrix cores by the loop of mfma_tiles.h, x [M, K], W [N, K] as the reference
// stores its linears' weights (ullm/layers/linear.py:165,268): a block takes 64 WMW rows of x against 256 rows of W.
//   store   bfloat16 [M, N], with an optional bias
//   gated   W holds gate rows, then as many up rows: bfloat16 [M, N / 2] of silu(gate) * up (or the clamped unit), a block taking
//           the gate and the up rows of 128 columns
//   float   the 32-bit sums themselves
//
// What bounds it is the matrix pipe and, over a long run, the power the chip may draw: 12 000 x 4096 x 12288 takes 896 us, 1.35
// PFLOP/s (the library 1160; 8192 x 8192 x 8192 in the library 1.37 PFLOP/s); then the last round of blocks, so it is taken where
// the tiles fill their rounds or the library's choice falls off (dispatch.limits and dispatch.gated_tile_groups, which name both sides' times).  The gated
// form writes half the columns and spares the activation kernel's pass (604 -> 467 us at 3000 x 24576 x 4096).  Two neighbouring
// 16 x 16 results leave as lines of 64 bytes a row: 8192 x 6144 x 4096 302 -> 293 us against lines of 32.
#include "mfma_tiles.h"
#include "launchers.h"

enum { TILES_STORE = 0, TILES_GATED = 1, TILES_FLOAT = 2 };

template <int WMW, int STAGES, int MODE>
__global__ void __launch_bounds__(128 * WMW)
gemm_tiles_kernel(const bf16_t* __restrict__ x, int ldx, const bf16_t* __restrict__ w, int ldw, const float* __restrict__ bias,
                  void* __restrict__ out_, int ldo, int M, int N, int K, int m_tiles, int n_tiles, float limit, float alpha) {
  using T = ProductTiles<WMW, STAGES>;
  extern __shared__ __attribute__((aligned(16))) unsigned char tile_stages[];
  // Blocks go to the chip's 8 dies round-robin by their id and every die has a second-level cache of its own: die d takes the
  // d-th eighth of the tiles, eight tiles of rows to a strip of W and strip after strip, so that what runs on a die at one time
  // is about a square of tiles
  const int total = m_tiles * n_tiles, per_die = (total + 7) / 8;
  const int item = ((int)blockIdx.x & 7) * per_die + ((int)blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_die || item >= total) return;
  const int band = item / (8 * n_tiles), in_band = item - band * 8 * n_tiles;
  const int rows_here = m_tiles - 8 * band < 8 ? m_tiles - 8 * band : 8;
  const int m0 = (8 * band + in_band % rows_here) * T::BM, nt = in_band / rows_here;
  constexpr bool GATED = MODE == TILES_GATED;
  constexpr int COLS = GATED ? 128 : 256;
  const int n_out = GATED ? N / 2 : N, n0 = nt * COLS;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  unsigned xoff[T::XL], woff[T::WL];
#pragma unroll
  for (int i = 0; i < T::XL; ++i) {
    const int row = T::x_row(wave, lane, i), m = m0 + row < M ? m0 + row : M - 1;
    xoff[i] = 2u * ((unsigned)m * (unsigned)ldx + T::k_of(row, lane));
  }
#pragma unroll
  for (int i = 0; i < T::WL; ++i) {
    const int row = T::w_row(wave, lane, i);
    int n = n0 + row % COLS;
    if (n >= n_out) n = n_out - 1;
    woff[i] = 2u * ((unsigned)((GATED && row >= COLS ? n_out : 0) + n) * (unsigned)ldw + T::k_of(row, lane));
  }
  tile_f32x4 acc[T::TN][T::TM];
  T::run(tile_stages, reinterpret_cast<const char*>(x), xoff, reinterpret_cast<const char*>(w), woff, K >> 6, 0, wave, lane, 128, acc);
  const int wm = wave >> 1, wn = wave & 1;
  const bool whole = ((n_out | ldo) & 7) == 0;
#pragma unroll
  for (int m = 0; m < T::TM; ++m) {
    const int row = m0 + 64 * wm + 16 * m + r;
    if (row >= M) continue;
#pragma unroll
    for (int n = 0; n < (GATED ? 4 : 8); n += 2) {
      const int c0 = n0 + 64 * wn + 16 * (n & 3) + (n < 4 ? 0 : 128);
      float v[2][4];
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int c = c0 + 16 * h + 4 * g + i;
          v[h][i] = acc[n + h][m][i];
          if constexpr (GATED) v[h][i] = gated_unit(v[h][i], acc[n + h + 4][m][i], limit, alpha);
          if (MODE == TILES_STORE && bias) v[h][i] += bias[c < n_out ? c : n_out - 1];
        }
      // n_out and ldo are multiples of four
      if constexpr (MODE == TILES_FLOAT) {
        float* const o = reinterpret_cast<float*>(out_) + (size_t)row * ldo;
#pragma unroll
        for (int h = 0; h < 2; ++h)
          if (c0 + 16 * h + 4 * g < n_out)
            *reinterpret_cast<float4*>(o + c0 + 16 * h + 4 * g) = make_float4(v[h][0], v[h][1], v[h][2], v[h][3]);
      } else {
        bf16_t* const o = reinterpret_cast<bf16_t*>(out_) + (size_t)row * ldo;
        const uint2 left = make_uint2(pack2_bf16(v[0][0], v[0][1]), pack2_bf16(v[0][2], v[0][3]));
        const uint2 right = make_uint2(pack2_bf16(v[1][0], v[1][1]), pack2_bf16(v[1][2], v[1][3]));
        if (whole) {
          const uint4 both = pair_columns(left, right);
          const int c = c0 + pair_column(g);
          if (c < n_out) *reinterpret_cast<uint4*>(o + c) = both;
        } else {
          const int c = c0 + 4 * g;
          if (c < n_out) *reinterpret_cast<uint2*>(o + c) = left;
          if (c + 16 < n_out) *reinterpret_cast<uint2*>(o + c + 16) = right;
        }
      }
    }
  }
}

template <int WMW, int STAGES, int MODE, typename... Args>
static int launch_tiles(long long blocks, hipStream_t stream, Args... args) {
  constexpr int bytes = ProductTiles<WMW, STAGES>::BYTES;
  static const hipError_t allowed = hipFuncSetAttribute((const void*)gemm_tiles_kernel<WMW, STAGES, MODE>,
                                                        hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (allowed != hipSuccess) return (int)allowed;
  hipLaunchKernelGGL((gemm_tiles_kernel<WMW, STAGES, MODE>), dim3((unsigned)(8 * ((blocks + 7) / 8))), dim3(128 * WMW), bytes, stream,
                     args...);
  ULLM_LAUNCH_CHECK();
}

// Whether the kernel takes the operands: rows whose ends 32-bit byte offsets reach, K in whole stages.
extern "C" int ullm_gemm_tiles_supports(int M, int N, int K, int ldx, int ldw, int mode) {
  return M >= 1 && K >= 64 && K % 64 == 0 && ldx % 8 == 0 && ldw % 8 == 0 && ldx >= K && ldw >= K && N % 4 == 0 &&
         (mode != TILES_GATED || N % 8 == 0) && (long long)M * ldx < (1LL << 31) && (long long)N * ldw < (1LL << 31);
}

// row_groups: 64-row groups a block takes (2 or 4).
extern "C" int ullm_gemm_tiles(const void* x, int ldx, const void* w, int ldw, const float* bias, void* out, int ldo, int M, int N,
                               int K, int mode, int row_groups, float limit, float alpha, hipStream_t stream) {
  if (M <= 0 || N <= 0) return 0;
  if (!ullm_gemm_tiles_supports(M, N, K, ldx, ldw, mode) || mode < TILES_STORE || mode > TILES_FLOAT) return ULLM_ERR_SHAPE;
  if (((uintptr_t)x | (uintptr_t)w | (uintptr_t)out) & 15 || ldo % 4 || ldo < (mode == TILES_GATED ? N / 2 : N)) return ULLM_ERR_SHAPE;
  const int bm = 64 * row_groups, mt = (M + bm - 1) / bm, nt = (N + 255) / 256;
  const long long total = (long long)mt * nt;
  if (total > 0x3fffffffLL) return ULLM_ERR_SHAPE;
#define GO(W, ST, MODE) return launch_tiles<W, ST, MODE>(total, stream, (const bf16_t*)x, ldx, (const bf16_t*)w, ldw, bias, out, ldo, M, N, \
    K, mt, nt, limit, alpha)
#define ROWS(W, ST) do { if (mode == TILES_STORE) GO(W, ST, TILES_STORE); if (mode == TILES_GATED) GO(W, ST, TILES_GATED); \
    GO(W, ST, TILES_FLOAT); } while (0)
  if (row_groups == 2) ROWS(2, 3);
  if (row_groups == 4) ROWS(4, 2);
#undef ROWS
#undef GO
  return ULLM_ERR_SHAPE;
}
