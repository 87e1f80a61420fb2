// The inner loop of large bfloat16 products out = x W^T: a block of WMW x WN waves takes 64 WMW rows of x against 256 rows of W,
// 64 values of K a stage.
//
// Stages go straight to shared memory (lds_load.h), STAGES of them taking turns: rows of 128 bytes, the 64 WMW rows of x and
// then the 256 of W, whose 16-byte piece c of row r lies at piece c ^ ((r >> 1) & 7) (the 16 lanes that shared memory serves
// together then read 16 different bank groups).  A load instruction fills 8 rows.  Wave (wm, wn) makes rows 64 wm .. of x
// against two strips of 128 / WN rows of W: with WN = 2 that is 12 reads of 1 KB per 32 products of v_mfma_f32_16x16x32_bf16, 96 of
// shared memory's 128 bytes a cycle at the matrix pipe's full rate.  WN = 8 is for eight waves over 64 rows of x.
//
// One wave's instructions keep the matrix pipe busy: the operands of one half of a stage (32 values of K) are read into
// registers between the products of the half before, and the loads of a stage further on are issued between the products of
// the second half, behind the one barrier of a stage, which stands where the operands of the half that follows it are in
// registers already.  With eight waves, two a unit, the reads stand beside the first six of a half's eight groups of products,
// so that they are back before the barrier, and a wave between its products lets the other go first: 8192 x 4096 x 12288 625 ->
// 564 us, 8192 x 6144 x 4096 303 -> 292 us; with four waves that order is 1 to 4 % slower.  Also tried at the first of these sizes:
// waves of 128 x 128 (one a unit) 725 us, products of 32 x 32 x 16 647 us, stages of 32 values of K, four or five of them, 618 us.
#pragma once
#include <type_traits>
#include "common.h"
#include "lds_load.h"

typedef __attribute__((ext_vector_type(8))) __bf16 tile_bf16x8;
typedef __attribute__((ext_vector_type(4))) float tile_f32x4;
union TilePack {
  tile_bf16x8 v;
  uint4 u4;
};

// A lane's packed bfloat16 values of two neighbouring 16 x 16 products (columns 4 g .. 4 g + 3 of each, a the left one's) as eight
// columns of one of them, from pair_column(g) of the left one's first on: whole lines of 64 bytes a row instead of halves.
__device__ __forceinline__ uint4 pair_columns(const uint2& a, const uint2& b) {
#ifdef __HIP_DEVICE_COMPILE__
  const auto p = __builtin_amdgcn_permlane16_swap(a.x, b.x, false, false);
  const auto q = __builtin_amdgcn_permlane16_swap(a.y, b.y, false, false);
  return make_uint4(p[0], q[0], p[1], q[1]);
#else
  return make_uint4(a.x, a.y, b.x, b.y);
#endif
}
__device__ __forceinline__ int pair_column(int g) { return 16 * (g & 1) + 4 * (g & 2); }

template <int WMW, int STAGES_, int WN = 2, bool TURNED_ = false>
struct ProductTiles {
  static constexpr bool TURNED = TURNED_;
  static constexpr int WAVES = WN * WMW, BM = 64 * WMW, BN = 256, STAGES = STAGES_, STAGE = (BM + BN) * 128;
  static_assert(WAVES == 4 || WAVES == 8, "whole pieces of x and of W a wave");
  static constexpr int XL = 8 / WN, WL = 32 / WAVES, LOADS = XL + WL, TM = 4, TN = 16 / WN, STRIP = TN / 2;
  static constexpr int BYTES = STAGES * STAGE;

  // row of x (of W) that this lane's i-th load brings, and the value of K in it
  static __device__ __forceinline__ int x_row(int wave, int lane, int i) { return 8 * (XL * wave + i) + (lane >> 3); }
  static __device__ __forceinline__ int w_row(int wave, int lane, int i) { return 8 * (WL * wave + i) + (lane >> 3); }
  static __device__ __forceinline__ int k_of(int row, int lane) { return 8 * ((lane & 7) ^ ((row >> 1) & 7)); }

  // xb, wb: addresses of K = 0 that the byte offsets xoff, woff count from; steps = K / 64 >= 1, of which (TURNED, else 0) the start-th
  // is the first and the one before it the last (where nobody turns, the count behind it costs 0.3 to 1.6 %: 512 x 24576 x 4096 gated 98.0 us and
  // 99.6, 12 000 rows 1703 and 1709); strip: rows between the two
  // strips of W that a wave takes (strip 0 begins at 16 STRIP wn of them).  acc[n][m]: lane (r, g) holds row 64 wm + 16 m + r of x,
  // rows 4 g .. 4 g + 3 of the n-th 16 rows of the wave's strips (n < STRIP: the first).
  static __device__ __forceinline__ void run(unsigned char* lds, const char* xb, const unsigned (&xoff)[XL], const char* wb,
                                             const unsigned (&woff)[WL], int steps, int start, int wave, int lane, int strip,
                                             tile_f32x4 (&acc)[TN][TM]) {
    int until_end = steps - start;
    if constexpr (TURNED) xb += start * 128, wb += start * 128;
    auto advance = [&]() __attribute__((always_inline)) {
      const bool wrap = TURNED && --until_end == 0;
      const int by = wrap ? 128 - 128 * steps : 128;
      xb += by, wb += by;
      if (wrap) until_end = steps;
    };
    const int r = lane & 15, g = lane >> 4, wm = wave / WN, wn = wave % WN;
    const unsigned place = lds_place(lds);
    const unsigned xdest = place + XL * wave * 1024, wdest = place + BM * 128 + WL * wave * 1024;
    auto load = [&](int i, unsigned to) __attribute__((always_inline)) {
      if (i < XL) load16_to_lds_from(xb, xoff[i], xdest + to + i * 1024);
      else load16_to_lds_from(wb, woff[i - XL], wdest + to + (i - XL) * 1024);
    };
    int at[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) at[s] = ((4 * s + g) ^ ((r >> 1) & 7)) << 4;
    const int xat = (64 * wm + r) * 128, wat = (BM + 16 * STRIP * wn + r) * 128, next = strip * 128;
    auto read_x = [&](const unsigned char* st, int s, int m) __attribute__((always_inline)) {
      return ld16(st + xat + at[s] + m * 2048);
    };
    auto read_w = [&](const unsigned char* st, int s, int n) __attribute__((always_inline)) {
      return ld16(st + wat + at[s] + n % STRIP * 2048 + (n < STRIP ? 0 : next));
    };
#pragma unroll
    for (int n = 0; n < TN; ++n)
#pragma unroll
      for (int m = 0; m < TM; ++m) acc[n][m] = tile_f32x4{0.f, 0.f, 0.f, 0.f};
    TilePack x[2][TM], w[2][TN];
    // the reads of half s that stand beside its predecessor's n-th group of products
    auto operands = [&](const unsigned char* st, int s, int n) __attribute__((always_inline)) {
      if constexpr (WAVES == 8) {
        constexpr int EACH = (TM + TN + TN - 1) / TN;
#pragma unroll
        for (int q = EACH * n; q < EACH * (n + 1); ++q) {
          if (q < TM) x[s][q].u4 = read_x(st, s, q);
          else if (q < TM + TN) w[s][q - TM].u4 = read_w(st, s, q - TM);
        }
      } else {
        if (n < TM) x[s][n].u4 = read_x(st, s, n);
        w[s][n].u4 = read_w(st, s, n);
      }
    };
    auto products = [&](int s, int n) __attribute__((always_inline)) {
      if constexpr (WAVES == 8) __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int m = 0; m < TM; ++m) acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[s][n].v, x[s][m].v, acc[n][m], 0, 0, 0);
      if constexpr (WAVES == 8) __builtin_amdgcn_s_setprio(0);
    };
#pragma unroll
    for (int i = 0; i < STAGES; ++i)
      if (i < steps) {
#pragma unroll
        for (int j = 0; j < LOADS; ++j) load(j, i * STAGE);
        advance();
      }
    if (steps >= STAGES) loads_left<(STAGES - 1) * LOADS>();
    else loads_left<0>();
    bare_barrier();
#pragma unroll
    for (int m = 0; m < TM; ++m) x[0][m].u4 = read_x(lds, 0, m);
#pragma unroll
    for (int n = 0; n < TN; ++n) w[0][n].u4 = read_w(lds, 0, n);
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
    // behind the wait and the barrier stage k + 1 is there (of this wave's loads only those of the stages behind it are left)
    // and no wave still reads stage k, whose place the loads then take
    auto second_half = [&](auto loads) __attribute__((always_inline)) {
      const unsigned to = buf * STAGE;
      buf = buf == STAGES - 1 ? 0 : buf + 1;
      const unsigned char* const nx = lds + buf * STAGE;
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
      if constexpr (decltype(loads)::value) advance();
    };
    int k = 0;
#pragma unroll 1
    for (; k + STAGES < steps; ++k) {
      first_half(lds + buf * STAGE);
      loads_left<(STAGES - 2) * LOADS>();
      bare_barrier();
      second_half(std::integral_constant<bool, true>{});
    }
#pragma unroll 1
    for (; k + 1 < steps; ++k) {
      first_half(lds + buf * STAGE);
      if (STAGES > 2 && k + 2 < steps) loads_left<(STAGES - 2) * LOADS>();
      else loads_left<0>();
      bare_barrier();
      second_half(std::integral_constant<bool, false>{});
    }
    first_half(lds + buf * STAGE);
#pragma unroll
    for (int n = 0; n < TN; ++n) products(1, n);
  }
};
