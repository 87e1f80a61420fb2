// Routed feed-forward (mixture of experts): routing, the grouping of (token, chosen expert) pairs by expert,
// the experts' two products over the grouped rows, and the weighted sum.  Nothing here waits for the device
// or sizes a launch by values: grids are made for the most tiles any routing can give, and a block whose
// tile is empty leaves at once, so a step can be captured into a graph.
//
//   route     logits [T, R] (R = experts with weights + identity experts) -> softmax over all R, the choice by
//             softmax + correction, the `top` largest (ties: the lower index), weights = the chosen experts'
//             softmax values over their sum (+ 1e-20).  Or (mode ROUTE_TOP_LOGITS) the `top` largest of logits +
//             bias, weights = the softmax over those alone.  Or (mode ROUTE_SIGMOID) scores = sigmoid(logit) each on
//             its own, the choice by score + correction, weights = the chosen scores over their sum (+ 1e-20).  The
//             weights are multiplied by one constant.  All 32-bit.  One wave per token.
//   sort      pairs (token, k) -> rows ("slots") grouped by expert; identity experts (index >= experts) get no
//             slot.  Which slot inside its expert a pair gets depends on timing; no value does: every row of a
//             product is a function of that row alone.  Also the tile list: (expert, first slot, rows <= tile_rows).
//   gate_up   act[slot, :] = glu(x[token of slot] Wg[e]^T, x Wu[e]^T) with the clamped gated unit
//             g' = min(g, limit), u' = clamp(u, -limit, limit), act = g' sigmoid(alpha g') (u' + 1),
//             or without a limit (limit <= 0) the plain unit silu(g) u
//   down      y[slot, :] = act[slot] Wd[e]^T, 32-bit
//   combine   out[t] = base[t] + bias + shared[t] + sum_k weight[t, k] * (expert k has weights ? y[slot(t, k)] : x[t]),
//             added in the order of k, 32-bit.
//
// Products: bfloat16 on v_mfma_f32_16x16x32_bf16 (A operand = 16 rows of an expert's matrix, lane (r, g) holds
// W[n0 + r][k + 8g .. +8]; B operand = 16 grouped rows of x; lane (r, g) then holds out[row r][column n0 + 4g .. +4]),
// or for float32 and for shapes the tiles do not take a kernel with one wave per output value that sums K in a
// fixed order.  Expert matrices are stacked: gate|up [experts, 2 ff, hidden], down [experts, hidden, ff].
#include "common.h"
#include "mfma_tiles.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
union Pack8 {
  bf16x8_t v;
  uint4 u4;
};

#define MOE_MAX_ROUTER 1024          // router outputs (experts + identity experts)
#define MOE_MAX_TOP 32

// ------------------------------------------------------------------------------- routing
// One wave: softmax over the logits z[0 .. n_router) in shared memory (overwritten by the scores), the `top` largest
// of score + correction, the chosen scores over their sum.  s_choice holds n_router floats, s_pick MOE_MAX_TOP.
// mode ROUTE_TOP_LOGITS: `correction` is a bias on the logits; the `top` largest of logit + bias are chosen and
// weighed by the softmax over the chosen ones alone.
// mode ROUTE_SIGMOID: every score is the sigmoid of its own logit; choice and weights as for ROUTE_SOFTMAX_ALL.
// Every weight is multiplied by `weight_scale`.  `raw`: the weights are the chosen scores as they are, not over their sum
// (not with ROUTE_TOP_LOGITS).  groups > 1: the outputs form that many equal groups of neighbours (at most 64), a group
// counts as much as the `group_top` (1 or 2) largest choice scores in it together, and only outputs of the `keep` best
// groups (ties: the lower index) can be chosen.
enum { ROUTE_SOFTMAX_ALL = 0, ROUTE_TOP_LOGITS = 1, ROUTE_SIGMOID = 2 };
__device__ __forceinline__ void route_from_logits(float* z, float* s_choice, float* s_pick,
                                                  const float* __restrict__ correction, int n_router, int top,
                                                  int* __restrict__ ids, float* __restrict__ weights, int lane,
                                                  int mode, float weight_scale, int groups, int keep, int raw, int group_top) {
  if (mode == ROUTE_TOP_LOGITS) {
    for (int e = lane; e < n_router; e += 64) {
      const float v = z[e] + (correction ? correction[e] : 0.f);
      z[e] = v;
      s_choice[e] = v;
    }
  } else if (mode == ROUTE_SIGMOID) {
    for (int e = lane; e < n_router; e += 64) {
      const float s = 1.f / (1.f + expf(-z[e]));
      z[e] = s;
      s_choice[e] = s + (correction ? correction[e] : 0.f);
    }
  } else {
    float mx = -INFINITY;
    for (int e = lane; e < n_router; e += 64) mx = fmaxf(mx, z[e]);
    mx = wave_max(mx);
    float sum = 0.f;
    for (int e = lane; e < n_router; e += 64) {
      const float p = expf(z[e] - mx);
      z[e] = p;
      sum += p;
    }
    sum = wave_sum(sum);
    for (int e = lane; e < n_router; e += 64) {
      const float s = z[e] / sum;
      z[e] = s;
      s_choice[e] = s + (correction ? correction[e] : 0.f);
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_wave_barrier();
  if (groups > 1) {
    const int size = n_router / groups;
    float mine = -INFINITY, next = -INFINITY;            // the group's two largest choice scores
    if (lane < groups)
      for (int j = 0; j < size; ++j) {
        const float c = s_choice[lane * size + j];
        next = fmaxf(next, fminf(mine, c));
        mine = fmaxf(mine, c);
      }
    if (group_top == 2 && size > 1) mine += next;
    int rank = 0;                                        // how many groups come before this lane's
    for (int o = 0; o < groups; ++o) {
      const float other = __shfl(mine, o, 64);
      if (other > mine || (other == mine && o < lane)) ++rank;
    }
    if (lane < groups && rank >= keep)
      for (int j = 0; j < size; ++j) s_choice[lane * size + j] = -INFINITY;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
  }
  float total = 0.f;
  for (int k = 0; k < top; ++k) {
    float best = -INFINITY;
    int at = 0x7fffffff;
    for (int e = lane; e < n_router; e += 64) {
      const float c = s_choice[e];
      if (c > best || (c == best && e < at)) {
        best = c;
        at = e;
      }
    }
    const float most = wave_max(best);
    at = wave_min(best == most ? at : 0x7fffffff);      // ties: the lower index
    if (at >= n_router) at = k < n_router ? k : 0;       // every value a NaN: any expert
    const float s = z[at];
    total += s;
    if (lane == 0) {
      ids[k] = at;
      s_pick[k] = s;
      s_choice[at] = -INFINITY;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_wave_barrier();
  }
  if (mode == ROUTE_TOP_LOGITS) {
    // the first pick is the largest: softmax over the picked logits, added in the order they were picked
    const float mx = s_pick[0];
    float sum = 0.f;
    for (int k = 0; k < top; ++k) sum += expf(s_pick[k] - mx);
    if (lane < top) weights[lane] = expf(s_pick[lane] - mx) / sum * weight_scale;
    return;
  }
  if (lane < top) weights[lane] = (raw ? s_pick[lane] : s_pick[lane] / (total + 1e-20f)) * weight_scale;
}

__global__ void __launch_bounds__(64)
moe_route_kernel(const float* __restrict__ logits, int ld, const float* __restrict__ correction, int n_router, int top,
                 int* __restrict__ ids, float* __restrict__ weights, int mode, float weight_scale, int groups, int keep, int raw, int group_top) {
  __shared__ float s_soft[MOE_MAX_ROUTER], s_choice[MOE_MAX_ROUTER];
  __shared__ float s_pick[MOE_MAX_TOP];
  const int t = blockIdx.x, lane = threadIdx.x;
  for (int e = lane; e < n_router; e += 64) s_soft[e] = logits[(size_t)t * ld + e];
  __syncthreads();
  route_from_logits(s_soft, s_choice, s_pick, correction, n_router, top, ids + (size_t)t * top, weights + (size_t)t * top, lane,
                    mode, weight_scale, groups, keep, raw, group_top);
}

static bool bad_groups(int n_router, int top, int mode, int groups, int keep, int raw, int group_top) {
  return groups < 1 || groups > 64 || keep < 1 || keep > groups || n_router % groups || top > n_router / groups * keep ||
         (raw && mode == ROUTE_TOP_LOGITS) || (group_top != 1 && group_top != 2);
}

extern "C" int ullm_moe_route(const float* logits, int ld, const float* correction, int T_, int n_router, int top,
                              int* ids, float* weights, int mode, float weight_scale, int groups, int keep, int raw,
                              int group_top, hipStream_t stream) {
  if (T_ <= 0) return 0;
  if (bad_groups(n_router, top, mode, groups, keep, raw, group_top)) return ULLM_ERR_SHAPE;
  if (n_router < 1 || n_router > MOE_MAX_ROUTER || top < 1 || top > MOE_MAX_TOP || top > n_router || ld < n_router)
    return ULLM_ERR_SHAPE;
  if (mode < ROUTE_SOFTMAX_ALL || mode > ROUTE_SIGMOID) return ULLM_ERR_UNSUPPORTED;
  hipLaunchKernelGGL(moe_route_kernel, dim3(T_), dim3(64), 0, stream, logits, ld, correction, n_router, top, ids, weights,
                     mode, weight_scale, groups, keep, raw, group_top);
  ULLM_LAUNCH_CHECK();
}

// The router's product and the routing in one kernel: a block of WAVES waves takes TPB tokens, whose rows lie in shared memory as
// they come; every wave takes U router outputs at a time with 16 / U 16-byte pieces of each of their rows a lane under way, and every
// piece fetched serves all the block's tokens.  A lane adds a token's pieces in rising order, then the wave adds up: an order
// that depends on nothing but the row.  Then wave v routes token v.  The router's matrix is 32-bit [n_router, H].
//
// What bounds it: few tokens by the chain of trips to memory, so the first pieces of the matrix are asked for behind the rows' first
// and before anything waits, the corrections too, and eight or sixteen waves take up to 32 or 64 outputs in one round; many
// tokens by the matrix's bytes from the second-level caches, 256 KB a block at 32 outputs of width 2048, and
// by multiply-adds.  Rows read two bytes a load by four waves, and four of sixteen waves' outputs a round, the matrix asked for behind
// them: 32 outputs of width 2048 for 48 / 512 / 1000 / 3000 tokens 12.0 -> 11.2, 25.8 -> 13.0, 26.2 -> 14.6, 28.2 -> 21.7 us, width 4096 13.3 -> 12.1,
// 18 -> 14.7, 29 -> 16.2, 71 -> 29; level for one to 300 tokens of 64 outputs and more, slower by 2 % at 256 outputs of width 1024 and 8000 tokens and
// at 300 of 640 and 5000; eight tokens a block 20.6 us at 2048 tokens of the first, 34 at 3000.
template <typename S>
__device__ __forceinline__ float4 router_values(const S* p);
template <> __device__ __forceinline__ float4 router_values<float>(const float* p) { return *reinterpret_cast<const float4*>(p); }
template <> __device__ __forceinline__ float4 router_values<bf16_t>(const bf16_t* p) {
  const uint2 u = *reinterpret_cast<const uint2*>(p);
  return make_float4(__uint_as_float(u.x << 16), __uint_as_float(u.x & 0xffff0000u), __uint_as_float(u.y << 16),
                     __uint_as_float(u.y & 0xffff0000u));
}
typedef __attribute__((ext_vector_type(4))) unsigned router_u32x4;
// 16 bytes of a row of T, kept as S: as they are or, bfloat16 values, widened
template <typename T, typename S>
__device__ __forceinline__ void keep_router_values(S* p, router_u32x4 v) {
  if constexpr (sizeof(S) == sizeof(T)) {
    *reinterpret_cast<router_u32x4*>(p) = v;
  } else {
    *reinterpret_cast<router_u32x4*>(p) = router_u32x4{v.x << 16, v.x & 0xffff0000u, v.y << 16, v.y & 0xffff0000u};
    *reinterpret_cast<router_u32x4*>(p + 4) = router_u32x4{v.z << 16, v.z & 0xffff0000u, v.w << 16, v.w & 0xffff0000u};
  }
}

// Waves a SIMD that the registers are held to, where more blocks a unit are worth more than loads under way; 0: as they come.  (256 outputs of width
// 1024, 8000 tokens by fours 148.6 -> 144.5 us, 32-bit rows 145.3 -> 147.3; 300 of width 640, 3000 32-bit rows by ones 95.2 -> 91.5.)
constexpr int router_waves(int tpb, int waves, bool early, bool widened) {
  return early ? 0 : tpb == 1 && waves == 8 ? 8 : tpb == 4 && waves == 4 && widened ? 6 : 0;
}
template <typename T, typename S, int TPB, int WAVES, bool EARLY>
__global__ void __launch_bounds__(64 * WAVES, (router_waves(TPB, WAVES, EARLY, sizeof(T) < sizeof(S))))
moe_router_kernel(const T* __restrict__ x, int ldx, const float* __restrict__ w, const float* __restrict__ correction,
                  int n_tokens, int H, int n_router, int top, int* __restrict__ ids, float* __restrict__ weights, int mode,
                  float weight_scale, int groups, int keep, int raw, int group_top) {
  extern __shared__ __attribute__((aligned(16))) unsigned char router_rows[];
  S* const xrow = reinterpret_cast<S*>(router_rows);                   // [TPB][H]
  constexpr int RCAP = TPB == 1 ? MOE_MAX_ROUTER : 256;                // router outputs the variant takes
  constexpr int U = 4, PJ = 4, NT = 64 * WAVES, PER16 = 16 / (int)sizeof(T), AHEAD = TPB == 1 ? 1 : 4;
  static_assert(WAVES >= TPB, "a wave routes a token");
  __shared__ float z[TPB][RCAP], s_choice[TPB][RCAP], s_correction[RCAP];
  __shared__ float s_pick[TPB][MOE_MAX_TOP];
  const int t0 = blockIdx.x * TPB, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const bool vec = (H & 3) == 0 && (((uintptr_t)w) & 15) == 0;
  const int pieces = H >> 2;
  float4 wv[U][PJ];
  // the wave's U rows of the matrix, the pieces p0 + 64 j of each
  auto ask = [&](int e0, int p0) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < PJ; ++j) {
      const int pj = p0 + 64 * j < pieces ? p0 + 64 * j : pieces - 1;
#pragma unroll
      for (int u = 0; u < U; ++u)
        wv[u][j] = *reinterpret_cast<const float4*>(w + (size_t)(e0 + u < n_router ? e0 + u : n_router - 1) * H + 4 * pj);
    }
  };
  auto token = [&](int q) { return (size_t)(t0 + q < n_tokens ? t0 + q : n_tokens - 1) * ldx; };
  const float own = correction && tid < n_router ? correction[tid] : 0.f;
  if (H % PER16 == 0 && ldx % PER16 == 0 && ((uintptr_t)x & 15) == 0) {
    const int row16 = H / PER16, all = TPB * row16;
    router_u32x4 held[AHEAD];
    auto rows = [&](int at) __attribute__((always_inline)) {
#pragma unroll
      for (int k = 0; k < AHEAD; ++k) {
        const int i = at + k * NT < all ? at + k * NT : all - 1;
        const int q = TPB == 1 ? 0 : i / row16;
        held[k] = *reinterpret_cast<const router_u32x4*>(x + token(q) + (size_t)(i - q * row16) * PER16);
      }
    };
    rows(tid);
    if (EARLY && vec) ask(U * wave, lane);
    for (int at = tid;;) {
#pragma unroll
      for (int k = 0; k < AHEAD; ++k)
        if (at + k * NT < all) keep_router_values<T, S>(xrow + (size_t)(at + k * NT) * PER16, held[k]);
      at += AHEAD * NT;
      if (at - tid >= all) break;
      rows(at);
    }
  } else {
    if (EARLY && vec) ask(U * wave, lane);
    for (int q = 0; q < TPB; ++q)
      for (int i = tid; i < H; i += NT) {
        if constexpr (sizeof(S) == sizeof(T)) xrow[q * H + i] = x[token(q) + i];
        else xrow[q * H + i] = ld_f32(x + token(q) + i);
      }
  }
  if (correction) {
    if (tid < n_router) s_correction[tid] = own;
    for (int e = tid + NT; e < n_router; e += NT) s_correction[e] = correction[e];
  }
  __syncthreads();
  for (int e0 = U * wave; e0 < n_router; e0 += U * WAVES) {
    float a[TPB][U];
#pragma unroll
    for (int q = 0; q < TPB; ++q)
#pragma unroll
      for (int u = 0; u < U; ++u) a[q][u] = 0.f;
    if (vec) {
      for (int p0 = lane; p0 < pieces; p0 += 64 * PJ) {
        if (!EARLY || e0 != U * wave || p0 != lane) ask(e0, p0);
#pragma unroll
        for (int j = 0; j < PJ; ++j) {
          if (p0 + 64 * j >= pieces) break;
#pragma unroll
          for (int q = 0; q < TPB; ++q) {
            const float4 xv = router_values<S>(xrow + q * H + 4 * (p0 + 64 * j));
#pragma unroll
            for (int u = 0; u < U; ++u)
              a[q][u] = fmaf(xv.w, wv[u][j].w, fmaf(xv.z, wv[u][j].z, fmaf(xv.y, wv[u][j].y, fmaf(xv.x, wv[u][j].x, a[q][u]))));
          }
        }
      }
    } else {
      for (int i = lane; i < H; i += 64) {
#pragma unroll
        for (int q = 0; q < TPB; ++q)
#pragma unroll
          for (int u = 0; u < U; ++u)
            a[q][u] = fmaf(ld_f32(xrow + q * H + i), w[(size_t)(e0 + u < n_router ? e0 + u : n_router - 1) * H + i], a[q][u]);
      }
    }
#pragma unroll
    for (int q = 0; q < TPB; ++q)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float sum = wave_sum(a[q][u]);
        if (lane == 0 && e0 + u < n_router) z[q][e0 + u] = sum;
      }
  }
  __syncthreads();
  if (wave < TPB && t0 + wave < n_tokens)
    route_from_logits(z[wave], s_choice[wave], s_pick[wave], correction ? s_correction : nullptr, n_router, top, ids + (size_t)(t0 + wave) * top,
                      weights + (size_t)(t0 + wave) * top, lane, mode, weight_scale, groups, keep, raw, group_top);
}

extern "C" int ullm_moe_router(const void* x, int ldx, const float* w, const float* correction, int T_, int H,
                               int n_router, int top, int* ids, float* weights, int mode, float weight_scale, int groups, int keep,
                               int raw, int group_top, int dtype, hipStream_t stream) {
  if (T_ <= 0) return 0;
  if (bad_groups(n_router, top, mode, groups, keep, raw, group_top)) return ULLM_ERR_SHAPE;
  if (mode < ROUTE_SOFTMAX_ALL || mode > ROUTE_SIGMOID) return ULLM_ERR_UNSUPPORTED;
  if (n_router < 1 || n_router > MOE_MAX_ROUTER || top < 1 || top > MOE_MAX_TOP || top > n_router || H < 1 || ldx < H ||
      (size_t)H * sizeof(float) > 48 * 1024)
    return ULLM_ERR_SHAPE;
  if (dtype != ULLM_F32 && dtype != ULLM_BF16) return ULLM_ERR_DTYPE;
#define GO(TT, SS, TPB, WAVES, EARLY) hipLaunchKernelGGL((moe_router_kernel<TT, SS, TPB, WAVES, EARLY>), dim3((T_ + TPB - 1) / TPB), dim3(64 * WAVES), \
    (size_t)H * sizeof(SS) * TPB, stream, (const TT*)x, ldx, w, correction, T_, H, n_router, top, ids, weights, mode, weight_scale, groups, \
    keep, raw, group_top)
#define GOT(TPB, WAVES, EARLY) do { \
    if (dtype == ULLM_F32) GO(float, float, TPB, WAVES, EARLY); \
    else if (TPB == 1 || H * TPB <= 8192) GO(bf16_t, float, TPB, WAVES, EARLY); \
    else if constexpr (TPB > 1) GO(bf16_t, bf16_t, TPB, WAVES, EARLY); } while (0)
  // Tokens a block, its waves, and whether the matrix is asked for before the rows are there (which takes the registers of two blocks'
  // waves), by what fills the chip; several tokens where their rows fit 32 KB of shared memory, as 32-bit values if they do, and their scores
  // beside them.  us on a matrix that is not cached, 1 token of 16 waves / 1 of 8 early / 1 of 8 / 2 of 8 early / 4 of 8 early / 4 of 4
  // early / 4 of 4.  32 outputs of width 2048: 48 tokens 11.6 / 10.8 / 11.4 / 11.8 / 13.5 / 16.0 / 21.0, 400 13.3 / 13.8 / 13.1 / 12.5 / 13.3 /
  // 15.5 / 20.4, 1000 22 / 22 / 20 / 18 / 14.3 / 16.5 / 21, 3000 46 / - / - / - / - / 21.5 / 22.8; 128 of 1024: 48 14.7 / 15.3 / 17.3 / 17.4 / 22 / 29 / 39,
  // 400 21 / 20 / 20 / 18 / 21 / 28 / 38, 1000 36 / 34 / 32 / 27 / 22 / 29 / 39, 3000 75 / - / - / - / - / 42 / 44, 8000 172 / - / - / - / - / 92 / 84;
  // 16 of 512: 48 7.5 / 8.2 / 7.6 / 9.2 / 10.1 / 10.2 / 9.2, 1000 11.2 / 13.1 / 8.3 / 12.1 / 9.7 / 9.2 / 9.4, 8000 56 / - / - / - / - / 21 / 17.  Width 5120,
  // where two fit: 24 outputs, 1000 tokens 28 by ones, 18 by twos, 8000 152 and 87.
  // Rows that end inside a piece come one value a load, which many waves hide.  1 of 16 waves / 1 of 8 / 2 of 8 / 4 of 4: 200 outputs of width 1282, 400
  // tokens 40 / 60 / 64 / 118, 700 58 / 60 / 65 / 118, 1500 95 / 93 / 68 / 120, 4000 203 / 193 / 157 / 123; 33 of 770, 1000 tokens 17 / 16 / 17 / 25,
  // 1500 23 / 22 / 18 / 27, 3000 38 / 34 / 32 / 27; 60 of 6002, 700 62 / 69 / - / -, 1000 83 / 72 / - / -.
  // One token a block because two do not fit: sixteen waves where outputs take many rounds (256 of width 7168 in 32 bits, 700 tokens 196 and in eight
  // 203, but 400, where the chip holds all blocks of eight, 134 and 115); 300 outputs of width 640, 3000 tokens 94 and 91, 512 25.8 and 27.0, of width
  // 2048 3000 tokens 242 and 250; 100 of width 600, 400 tokens 12.4 and 13.2.
  const int most = n_router > 256 ? 1 : 32768 / (H * (dtype == ULLM_F32 ? 4 : 2));
  if (H % 4 || ((uintptr_t)w & 15)) {
    if (T_ > 1024 && most >= 4 && (T_ > 2048 || H <= 512)) GOT(4, 4, false);
    else if (T_ > 1024 && most >= 2) GOT(2, 8, false);
    else if (T_ > (H <= 2048 ? 512 : 800) && most >= 2) GOT(1, 8, false);
    else GOT(1, 16, false);
  } else if (T_ > 1024 && most >= 4) {
    if (H <= 512 || (H <= 1024 && T_ > 4096)) GOT(4, 4, false);
    else GOT(4, 4, true);
  } else if (T_ > 512 && most >= 4 && H >= 1024) GOT(4, 8, true);
  else if (T_ > 512 && most >= 2 && H >= 1024) GOT(2, 8, false);
  else if ((T_ > 300 || (T_ > 256 && H > 2048)) && most >= 2 && H >= 1024) GOT(2, 8, true);
  else if (n_router > 256 ? T_ > 512 && H <= 1024 : T_ > 512 ? H < 1024 || n_router <= 64 : T_ > 300 && (H >= 1024 || n_router <= 32)) GOT(1, 8, false);
  else if (T_ <= 300 && n_router <= 32 && H >= 2048) GOT(1, 8, true);
  else GOT(1, 16, false);
#undef GOT
#undef GO
  ULLM_LAUNCH_CHECK();
}

// ------------------------------------------------------------------------------- grouping by expert
// One block, bound by its trips to memory and shared memory: the first 16384 pairs are read once and counted with the addition that
// gives a pair its place, the running sums over the experts are one wave's (2048 tokens of 4 choices among 32 experts 7.6 -> 6.0 us,
// 3000 9.8 -> 7.5).  Pairs behind those are read twice, to be counted and to take their places (96000 pairs among 128 experts 68 us;
// with their places kept in slot_of_pair from the count on 79, as it took them all before 75).  offsets [experts + 1]; slot_of_pair [pairs] (-1: the pair's expert has no weights); token_of_slot [pairs];
// tiles [max_tiles + 1][3] = (expert, first slot, rows), rows 0 for the tiles no expert filled; the entry behind the
// list holds the number of tiles in use.
__global__ void __launch_bounds__(1024)
moe_sort_kernel(const int* __restrict__ ids, int n_pairs, int top, int n_experts, int tile_rows,
                int* __restrict__ offsets, int* __restrict__ slot_of_pair, int* __restrict__ token_of_slot,
                int* __restrict__ tiles, int max_tiles) {
  constexpr int HELD = 16;
  __shared__ int count[MOE_MAX_ROUTER], start[MOE_MAX_ROUTER + 1], tile_base[MOE_MAX_ROUTER + 1], taken[MOE_MAX_ROUTER];
  const int tid = threadIdx.x;
  for (int e = tid; e < n_experts; e += blockDim.x) count[e] = 0;
  __syncthreads();
  // a pair's place inside its expert is what the count held before it; the first HELD pairs of a thread keep theirs in registers
  int held_e[HELD], held_at[HELD];
#pragma unroll
  for (int i = 0; i < HELD; ++i) {
    const int p = tid + i * (int)blockDim.x;
    held_e[i] = p < n_pairs ? ids[p] : -1;
  }
#pragma unroll
  for (int i = 0; i < HELD; ++i) {
    if (held_e[i] >= n_experts) held_e[i] = -1;
    held_at[i] = held_e[i] >= 0 ? atomicAdd(&count[held_e[i]], 1) : 0;
  }
  // the pairs behind those come after them: counted here, given their places below
  if (n_pairs > HELD * (int)blockDim.x) {
    __syncthreads();
    for (int e = tid; e < n_experts; e += blockDim.x) taken[e] = count[e];
    __syncthreads();
    for (int p = tid + HELD * (int)blockDim.x; p < n_pairs; p += blockDim.x) {
      const int e = ids[p];
      if (e >= 0 && e < n_experts) atomicAdd(&count[e], 1);
    }
  }
  __syncthreads();
  if (tid < 64) {                                         // one wave: running sums over the experts, 64 at a time
    int off = 0, tb = 0;
    for (int e0 = 0; e0 < n_experts; e0 += 64) {
      const int e = e0 + tid, n = e < n_experts ? count[e] : 0;
      int a = n, b = (n + tile_rows - 1) / tile_rows;
      const int own_tiles = b;
#pragma unroll
      for (int m = 1; m < 64; m <<= 1) {
        const int pa = __shfl_up(a, m, 64), pb = __shfl_up(b, m, 64);
        if (tid >= m) {
          a += pa;
          b += pb;
        }
      }
      if (e < n_experts) {
        start[e] = off + a - n;
        tile_base[e] = tb + b - own_tiles;
      }
      off += __shfl(a, 63, 64);
      tb += __shfl(b, 63, 64);
    }
    if (tid == 0) {
      start[n_experts] = off;
      tile_base[n_experts] = tb;
    }
  }
  __syncthreads();
  for (int e = tid; e <= n_experts; e += blockDim.x) offsets[e] = start[e];
#pragma unroll
  for (int i = 0; i < HELD; ++i) {
    const int p = tid + i * (int)blockDim.x;
    if (p >= n_pairs) break;
    const int slot = held_e[i] >= 0 ? start[held_e[i]] + held_at[i] : -1;
    if (slot >= 0) token_of_slot[slot] = p / top;
    slot_of_pair[p] = slot;
  }
  for (int p = tid + HELD * (int)blockDim.x; p < n_pairs; p += blockDim.x) {
    const int e = ids[p];
    int slot = -1;
    if (e >= 0 && e < n_experts) {
      slot = start[e] + atomicAdd(&taken[e], 1);
      token_of_slot[slot] = p / top;
    }
    slot_of_pair[p] = slot;
  }
  for (int e = tid; e < n_experts; e += blockDim.x) {
    const int first = tile_base[e], n = tile_base[e + 1] - first;
    for (int i = 0; i < n && first + i < max_tiles; ++i) {
      const int left = count[e] - i * tile_rows;
      tiles[3 * (first + i)] = e;
      tiles[3 * (first + i) + 1] = start[e] + i * tile_rows;
      tiles[3 * (first + i) + 2] = left < tile_rows ? left : tile_rows;
    }
  }
  for (int i = tile_base[n_experts] + tid; i < max_tiles; i += blockDim.x) {
    tiles[3 * i] = 0;
    tiles[3 * i + 1] = 0;
    tiles[3 * i + 2] = 0;
  }
  if (tid == 0) {                                         // one more entry behind the list: how many tiles are in use
    tiles[3 * max_tiles] = tile_base[n_experts] < max_tiles ? tile_base[n_experts] : max_tiles;
    tiles[3 * max_tiles + 1] = 0;
    tiles[3 * max_tiles + 2] = 0;
  }
}

extern "C" int ullm_moe_sort(const int* ids, int n_pairs, int top, int n_experts, int tile_rows, int* offsets,
                             int* slot_of_pair, int* token_of_slot, int* tiles, int max_tiles, hipStream_t stream) {
  if (n_pairs <= 0) return 0;
  if (n_experts < 1 || n_experts > MOE_MAX_ROUTER || top < 1 || tile_rows < 1 || max_tiles < 1) return ULLM_ERR_SHAPE;
  // every routing fits: sum over experts of ceil(count / tile_rows) <= pairs / tile_rows + experts in use
  const long long most = (long long)n_pairs / tile_rows + (n_experts < n_pairs ? n_experts : n_pairs);
  if (max_tiles < most) return ULLM_ERR_SHAPE;
  hipLaunchKernelGGL(moe_sort_kernel, dim3(1), dim3(1024), 0, stream, ids, n_pairs, top, n_experts, tile_rows, offsets,
                     slot_of_pair, token_of_slot, tiles, max_tiles);
  ULLM_LAUNCH_CHECK();
}

// ------------------------------------------------------------------------------- the clamped gated unit
// limit <= 0: the plain gated unit silu(g) * u.
template <bool EXACT>
__device__ __forceinline__ float moe_glu(float g, float u, float limit, float alpha) {
  if (limit <= 0.f)
    return (EXACT ? g / (1.f + expf(-g)) : fast_silu(g)) * u;
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  const float sg = EXACT ? 1.f / (1.f + expf(-alpha * g))
                         : __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-1.4426950408889634f * alpha * g));
  return g * sg * (u + 1.f);
}

// ------------------------------------------------------------------------------- products, one wave per value
// grid (tiles, column blocks); a block of 4 waves takes one tile's rows in turn, the row of x in shared memory,
// and each wave its share of the block's columns: lanes stride K, then the wave adds up (a fixed order).
template <typename T, bool GATED>
__global__ void __launch_bounds__(256)
moe_rows_simple_kernel(const T* __restrict__ x, int ldx, const int* __restrict__ row_index,
                       const T* __restrict__ w, const int* __restrict__ tiles, void* __restrict__ out_, int ldo,
                       int n_out, int K, int cols_per_block, float limit, float alpha) {
  extern __shared__ float xrow[];
  const int tile = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int e = tiles[3 * tile], slot0 = tiles[3 * tile + 1], rows = tiles[3 * tile + 2];
  if (rows <= 0) return;
  const int c0 = blockIdx.y * cols_per_block;
  const int c1 = c0 + cols_per_block < n_out ? c0 + cols_per_block : n_out;
  const size_t w_rows = GATED ? 2 * (size_t)n_out : (size_t)n_out;
  const T* we = w + (size_t)e * w_rows * K;
  for (int r = 0; r < rows; ++r) {
    const int slot = slot0 + r;
    const T* xr = x + (size_t)(row_index ? row_index[slot] : slot) * ldx;
    __syncthreads();
    for (int i = tid; i < K; i += 256) xrow[i] = ld_f32(xr + i);
    __syncthreads();
    for (int c = c0 + wave; c < c1; c += 4) {
      const T* wg = we + (size_t)c * K;
      float a = 0.f, b = 0.f;
      for (int i = lane; i < K; i += 64) {
        a = fmaf(xrow[i], ld_f32(wg + i), a);
        if (GATED) b = fmaf(xrow[i], ld_f32(wg + (size_t)n_out * K + i), b);
      }
      a = wave_sum(a);
      if (GATED) b = wave_sum(b);
      if (lane == 0) {
        if (GATED) st_f32(reinterpret_cast<T*>(out_) + (size_t)slot * ldo + c, moe_glu<sizeof(T) == 4>(a, b, limit, alpha));
        else reinterpret_cast<float*>(out_)[(size_t)slot * ldo + c] = a;
      }
    }
  }
}

// Lane (r, g): row r of each 16-row group, columns c .. c + 3.
template <int MT, bool GATED>
__device__ __forceinline__ void moe_store_rows(const f32x4_t (&acc_g)[MT], const f32x4_t (&acc_u)[MT], void* out_, int ldo, int slot0,
                                               int rows, int c, int r, int n_out, float limit, float alpha) {
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int row = 16 * t + r;
    if (row >= rows) continue;
    const size_t at = (size_t)(slot0 + row) * ldo + c;
    if (GATED) {
      bf16_t* o = reinterpret_cast<bf16_t*>(out_) + at;
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = moe_glu<false>(acc_g[t][i], acc_u[t][i], limit, alpha);
      if (c + 3 < n_out && (ldo & 3) == 0) {
        *reinterpret_cast<uint2*>(o) = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (c + i < n_out) o[i] = f32_to_bf16_bits(v[i]);
      }
    } else {
      float* o = reinterpret_cast<float*>(out_) + at;
      if (c + 3 < n_out && (ldo & 3) == 0) {
        *reinterpret_cast<float4*>(o) = make_float4(acc_g[t][0], acc_g[t][1], acc_g[t][2], acc_g[t][3]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (c + i < n_out) o[i] = acc_g[t][i];
      }
    }
  }
}

// ------------------------------------------------------------------------------- products on the matrix cores
// Few rows a tile (single tokens of a step): grid (tiles, groups of 16 output columns); tile = up to 16 * MT grouped
// rows of one expert.  The block's four waves share the 16 columns (GATED: the 16 gate rows and the 16 up rows of
// those columns) and take every fourth step of 64 along K, two steps of 32 in flight each; their sums are added
// through shared memory in wave order.  The work is streaming the chosen experts' matrices once, so it is cut into
// many blocks with many loads under way.  No load stands under a condition: a row past the tile's reads its last
// row, a column past the end the last column, a piece past the end of K the row's last piece (and is replaced by
// zeros); none is stored.
template <int MT, bool GATED>
__global__ void __launch_bounds__(256)
moe_rows_mfma_kernel(const bf16_t* __restrict__ x, int ldx, const int* __restrict__ row_index,
                     const bf16_t* __restrict__ w, const int* __restrict__ tiles, void* __restrict__ out_, int ldo,
                     int n_out, int K, float limit, float alpha) {
  constexpr int VALS = (GATED ? 8 : 4) * MT;
  __shared__ float part[3][VALS][64];
  const int tile = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4;
  const int e = tiles[3 * tile], slot0 = tiles[3 * tile + 1], rows = tiles[3 * tile + 2];
  if (rows <= 0) return;
  const int n0 = blockIdx.y * 16;
  const size_t w_rows = GATED ? 2 * (size_t)n_out : (size_t)n_out;
  const int wrow = n0 + r < n_out ? n0 + r : n_out - 1;
  const bf16_t* wg = w + ((size_t)e * w_rows + wrow) * K;
  const bf16_t* wu = wg + (size_t)n_out * K;
  const bf16_t* xr[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int row = 16 * t + r < rows ? 16 * t + r : rows - 1;
    xr[t] = x + (size_t)(row_index ? row_index[slot0 + row] : slot0 + row) * ldx;
  }
  f32x4_t acc_g[MT], acc_u[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    acc_g[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    acc_u[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  const int last_piece = K - 8;                          // K is a multiple of 8
  const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
  for (int k0 = 64 * wave; k0 < K; k0 += 256) {
    Pack8 a_g[2], a_u[2], b[2][MT];
    bool in[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int k = k0 + 32 * s + 8 * g;
      in[s] = k <= last_piece;
      const int kk = in[s] ? k : last_piece;
      a_g[s].u4 = ld_stream16(wg + kk);
      if (GATED) a_u[s].u4 = ld_stream16(wu + kk);
#pragma unroll
      for (int t = 0; t < MT; ++t) b[s][t].u4 = ld16(xr[t] + kk);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        if (!in[s]) b[s][t].u4 = zero;
        acc_g[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_g[s].v, b[s][t].v, acc_g[t], 0, 0, 0);
        if (GATED) acc_u[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_u[s].v, b[s][t].v, acc_u[t], 0, 0, 0);
      }
    }
  }
  // the waves' sums, added in wave order
  if (wave > 0) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        part[wave - 1][(GATED ? 8 : 4) * t + i][lane] = acc_g[t][i];
        if (GATED) part[wave - 1][8 * t + 4 + i][lane] = acc_u[t][i];
      }
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int v = 0; v < 3; ++v)
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc_g[t][i] += part[v][(GATED ? 8 : 4) * t + i][lane];
        if (GATED) acc_u[t][i] += part[v][8 * t + 4 + i][lane];
      }
  moe_store_rows<MT, GATED>(acc_g, acc_u, out_, ldo, slot0, rows, n0 + 4 * g, r, n_out, limit, alpha);
}

// The same where K is a multiple of 64 and at least 256: a wave takes a run of K of its own (a quarter), so that it reads each
// of the block's rows of the matrix in one piece, and its stages of 64 values (16 or, gated, 32 rows of the matrix and the tile's
// rows of x, whole lines of 128 bytes) go straight to shared memory of its own, two taking turns (lds_load.h): no barrier, and
// nothing but addresses in registers while 8 to 16 KB a wave are on their way.  What bounds it is the experts' matrices from
// memory (gate|up of 32 experts, width 2048, 1024 columns: 268 MB, 43 us).  The kernel above asks for 64 bytes of a row at a time
// and holds them in registers; gate|up + down at 8 / 48 / 100 tokens, 4 experts each, 41 + 19 / 61 + 33 / 80 + 44 us
// there, 28 + 15 / 41 + 22 / 50 + 30 us here.  The matrices' loads do not stay in the caches: without that 32 + 14 / 50 + 29 / 54 + 33,
// and the kernels around this one found their smaller matrices and rows gone (the router 12.5 against 10.2 us at one token).
// Three stages, and a block less on each compute unit, were 1 to 4 % slower, and a third with tiles of 32 rows.
template <int MT, bool GATED>
__global__ void __launch_bounds__(256)
moe_rows_dma_kernel(const bf16_t* __restrict__ x, int ldx, const int* __restrict__ row_index,
                    const bf16_t* __restrict__ w, const int* __restrict__ tiles, void* __restrict__ out_, int ldo,
                    int n_out, int K, float limit, float alpha) {
  constexpr int VALS = (GATED ? 8 : 4) * MT, WR = GATED ? 32 : 16, ROWS = WR + 16 * MT, LOADS = ROWS / 8, STAGE = ROWS * 128;
  extern __shared__ __attribute__((aligned(16))) unsigned char row_stages[];
  const int tile = blockIdx.x, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int e = tiles[3 * tile], slot0 = tiles[3 * tile + 1], rows = tiles[3 * tile + 2];
  if (rows <= 0) return;
  const int n0 = blockIdx.y * 16;
  const size_t w_rows = GATED ? 2 * (size_t)n_out : (size_t)n_out;
  const int stages = K >> 6, s0 = stages * wave / 4, s1 = stages * (wave + 1) / 4;
  // an instruction of 64 lanes fills 8 rows of a stage; piece c of row r lies at piece c ^ ((r >> 1) & 7)
  const bf16_t* src[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int row = 8 * i + (lane >> 3), piece = 8 * ((lane & 7) ^ ((row >> 1) & 7));
    if (i < WR / 8) {
      const int n = n0 + (row & 15) < n_out ? n0 + (row & 15) : n_out - 1;
      src[i] = w + ((size_t)e * w_rows + (row >= 16 ? n_out : 0) + n) * K + 64 * s0 + piece;
    } else {
      const int m = row - WR < rows ? row - WR : rows - 1;
      src[i] = x + (size_t)(row_index ? row_index[slot0 + m] : slot0 + m) * ldx + 64 * s0 + piece;
    }
  }
  unsigned char* const mine = row_stages + 2 * STAGE * wave;
  auto fetch = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      if (i < WR / 8) load16_to_lds_once(src[i], mine + buf * STAGE + i * 1024);
      else load16_to_lds(src[i], mine + buf * STAGE + i * 1024);
      src[i] += 64;
    }
  };
  f32x4_t acc_g[MT], acc_u[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    acc_g[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    acc_u[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  const int n_stages = s1 - s0;                          // at least one
  for (int i = 0; i < 2 && i < n_stages; ++i) fetch(i);
  int buf = 0;
  for (int k = 0; k < n_stages; ++k) {
    if (k + 1 < n_stages) loads_left<LOADS>();           // those of the stage behind this one
    else loads_left<0>();
    const unsigned char* const st = mine + buf * STAGE;
    Pack8 a_g[2], a_u[2], b[2][MT];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int at = r * 128 + (((4 * s + g) ^ ((r >> 1) & 7)) << 4);
      a_g[s].u4 = ld16(st + at);
      if (GATED) a_u[s].u4 = ld16(st + 2048 + at);
#pragma unroll
      for (int t = 0; t < MT; ++t) b[s][t].u4 = ld16(st + WR * 128 + t * 2048 + at);
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        acc_g[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_g[s].v, b[s][t].v, acc_g[t], 0, 0, 0);
        if (GATED) acc_u[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a_u[s].v, b[s][t].v, acc_u[t], 0, 0, 0);
      }
    if (k + 2 < n_stages) {
      reads_done();
      fetch(buf);
    }
    buf ^= 1;
  }
  // the waves' sums, added in wave order (no wave reads a stage any more)
  __syncthreads();
  float (*const part)[VALS][64] = reinterpret_cast<float (*)[VALS][64]>(row_stages);
  if (wave > 0) {
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        part[wave - 1][(GATED ? 8 : 4) * t + i][lane] = acc_g[t][i];
        if (GATED) part[wave - 1][8 * t + 4 + i][lane] = acc_u[t][i];
      }
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int v = 0; v < 3; ++v)
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc_g[t][i] += part[v][(GATED ? 8 : 4) * t + i][lane];
        if (GATED) acc_u[t][i] += part[v][8 * t + 4 + i][lane];
      }
  moe_store_rows<MT, GATED>(acc_g, acc_u, out_, ldo, slot0, rows, n0 + 4 * g, r, n_out, limit, alpha);
}

// Many rows a tile (prompt portions): a block per (tile, 128 rows of the expert's matrix); tile = up to 16 MT = 64 or 128
// grouped rows of one expert.  A stage is 64 values of K: the tile's rows of x and 128 rows of the matrix (GATED: the
// gate rows and the up rows of 64 output columns; else 128 output columns) go through shared memory once a block,
// 128-byte rows whose 16-byte piece c of row r lies at piece c ^ ((r >> 1) & 7) (the 16 lanes the hardware serves
// together then read 16 different bank groups); the next stage is fetched into registers while the products of this
// one run.  Wave v takes matrix rows 16 v .. and 64 + 16 v .. (GATED: gate and up of the same columns) against all
// rows of x: 16 products per 12 reads of shared memory at 64 rows, 32 per 20 at 128 (and 64 rather than 43 products
// per byte fetched).
template <int MT, bool GATED>
__global__ void __launch_bounds__(256)
moe_tiles_mfma_kernel(const bf16_t* __restrict__ x, int ldx, const int* __restrict__ row_index,
                      const bf16_t* __restrict__ w, const int* __restrict__ tiles, int n_tiles, int n_col_blocks,
                      void* __restrict__ out_, int ldo, int n_out, int K, float limit, float alpha) {
  extern __shared__ __attribute__((aligned(16))) unsigned char tile_stages[];  // two stages take turns: x, then the matrix
  constexpr int XB = 16 * MT * 128, WB = 128 * 128;
  unsigned char* const xs2[2] = {tile_stages, tile_stages + XB + WB};
  unsigned char* const ws2[2] = {tile_stages + XB, tile_stages + 2 * XB + WB};
  // Workgroups go to the chip's 8 dies round-robin by their id and every die has a second-level cache of its own:
  // die d takes the d-th eighth of the tiles in use, tile by tile in the list's order with all of a tile's column
  // blocks side by side.  What runs on a die at one time is then a few tiles of one or two experts: a tile's rows
  // of x are fetched once for all its column blocks, an expert's matrix once for all its tiles.
  const int used = tiles[3 * n_tiles];
  const int total = used * n_col_blocks, per_die = (total + 7) / 8;
  const int item = ((int)blockIdx.x & 7) * per_die + ((int)blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_die || item >= total) return;
  const int tile = item / n_col_blocks, col_block = item % n_col_blocks;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, g = lane >> 4;
  const int e = tiles[3 * tile], slot0 = tiles[3 * tile + 1], rows = tiles[3 * tile + 2];
  if (rows <= 0) return;
  const int cols = GATED ? 64 : 128;                      // output columns of a block
  const int n0 = col_block * cols;
  const size_t w_rows = GATED ? 2 * (size_t)n_out : (size_t)n_out;
  const bf16_t* we = w + (size_t)e * w_rows * K;
  // what this thread fetches of a stage: piece `pc` of x rows prow + 32 i and of matrix rows prow + 32 i
  constexpr int XP = MT / 2;                              // pieces of x a thread fetches a stage
  const int pc = tid & 7, prow = tid >> 3;
  const bf16_t* xsrc[XP];
  const bf16_t* wsrc[4];
  int xput[XP], wput[4];
#pragma unroll
  for (int i = 0; i < XP; ++i) {
    const int row = prow + 32 * i, rr = row < rows ? row : rows - 1;
    xsrc[i] = x + (size_t)(row_index ? row_index[slot0 + rr] : slot0 + rr) * ldx;
    xput[i] = row * 128 + ((pc ^ ((row >> 1) & 7)) << 4);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = prow + 32 * i;                       // 0 .. 127 of the block's matrix rows
    int n = GATED ? n0 + (row & 63) : n0 + row;
    if (n >= n_out) n = n_out - 1;
    wsrc[i] = we + ((GATED && row >= 64 ? (size_t)n_out : 0) + n) * K;
    wput[i] = row * 128 + ((pc ^ ((row >> 1) & 7)) << 4);
  }
  const int last_piece = K - 8;
  const uint4 zero = make_uint4(0u, 0u, 0u, 0u);
  // two sets of registers: a stage is fetched two stages before its products, written to shared memory one before
  uint4 xreg[2][XP], wreg[2][4];
  auto fetch = [&](int set, int k0) __attribute__((always_inline)) {
    const int k = k0 + 8 * pc;
    const bool in = k <= last_piece;
    const int kk = in ? k : last_piece;
#pragma unroll
    for (int i = 0; i < XP; ++i) xreg[set][i] = ld16(xsrc[i] + kk);
#pragma unroll
    for (int i = 0; i < 4; ++i) wreg[set][i] = ld16(wsrc[i] + kk);    // the expert's other tiles read the same rows: cached
    if (!in) {
#pragma unroll
      for (int i = 0; i < XP; ++i) xreg[set][i] = zero;
    }
  };
  auto put = [&](int set, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < XP; ++i) st16(xs2[buf] + xput[i], xreg[set][i]);
#pragma unroll
    for (int i = 0; i < 4; ++i) st16(ws2[buf] + wput[i], wreg[set][i]);
  };
  f32x4_t acc[2][MT];
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[h][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto products = [&](int buf) __attribute__((always_inline)) {
    const unsigned char* xs = xs2[buf];
    const unsigned char* ws = ws2[buf];
    // both steps of 32 are read before the first product: the second step's reads travel during the first's products
    Pack8 a[2][2], b[2][MT];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int row = 64 * h + 16 * wave + r;
        a[s][h].u4 = ld16(ws + row * 128 + (((4 * s + g) ^ ((row >> 1) & 7)) << 4));
      }
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        const int row = 16 * t + r;
        b[s][t].u4 = ld16(xs + row * 128 + (((4 * s + g) ^ ((row >> 1) & 7)) << 4));
      }
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < MT; ++t)
          acc[h][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[s][h].v, b[s][t].v, acc[h][t], 0, 0, 0);
  };
  // No fetch stands under a condition (the compiler then waits for every load under way at the next use of any): a
  // stage past the end of K reads the rows' last pieces again and is never written to shared memory.
  fetch(0, 0);
  put(0, 0);
  __syncthreads();
  fetch(0, 64);
  for (int k0 = 0; k0 < K; k0 += 128) {
    // stage k0 lies in buffer 0, set 0 holds stage k0 + 64 (on its way)
    fetch(1, k0 + 128);
    products(0);
    if (k0 + 64 < K) put(0, 1);          // buffer 1 was last read before the barrier that ended the step before
    __syncthreads();
    if (k0 + 64 >= K) break;
    // stage k0 + 64 lies in buffer 1, set 1 holds stage k0 + 128
    fetch(0, k0 + 192);
    products(1);
    if (k0 + 128 < K) put(1, 0);
    __syncthreads();
  }
  // lane (r, g): row r of each 16-row group; columns 16 wave + 4g .. + 4 of the block's (and 64 further on)
#pragma unroll
  for (int t = 0; t < MT; ++t) {
    const int row = 16 * t + r;
    if (row >= rows) continue;
    if (GATED) {
      const int c = n0 + 16 * wave + 4 * g;
      bf16_t* o = reinterpret_cast<bf16_t*>(out_) + (size_t)(slot0 + row) * ldo + c;
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = moe_glu<false>(acc[0][t][i], acc[1][t][i], limit, alpha);
      if (c + 3 < n_out && (ldo & 3) == 0) {
        *reinterpret_cast<uint2*>(o) = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (c + i < n_out) o[i] = f32_to_bf16_bits(v[i]);
      }
    } else {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int c = n0 + 64 * h + 16 * wave + 4 * g;
        float* o = reinterpret_cast<float*>(out_) + (size_t)(slot0 + row) * ldo + c;
        if (c + 3 < n_out && (ldo & 3) == 0) {
          *reinterpret_cast<float4*>(o) = make_float4(acc[h][t][0], acc[h][t][1], acc[h][t][2], acc[h][t][3]);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (c + i < n_out) o[i] = acc[h][t][i];
        }
      }
    }
  }
}

// The same products where K is a multiple of 64, by the loop of mfma_tiles.h: a block takes a tile of rows against 256 rows of the
// expert's matrix (GATED: the gate rows and the up rows of 128 output columns, a wave the same number of each).  Tiles of up to 128
// rows have four waves, tiles of up to 256 eight, which take 64 or 256 rows by 256, whichever holds the tile: an expert's
// short last tile is paid by its rows.  (128 rows by waves of their own, 64 by 64 each: 800 tokens gate|up + down 72 -> 70 us alone, but more reads of
// shared memory a product, and prompts of 3000 tokens in 4.29 ms instead of 4.27.)
// What bounds it: the experts' matrices from memory (268 MB of gate|up: 45 us) and, beside them, the matrix pipe, which the
// loop keeps busy 57 % of the time where every operand lies in the second-level cache.  Rows of the matrices lie a power of two apart, and
// blocks in step ask the same memory channels: so a block's K begins at the stage of its expert's number (where K is TURNED_K and more; 32 experts, width 2048, 1024
// columns, gate|up + down at 400 / 800 tokens, top 4, 71 + 26 / 73 + 35 -> 50 + 27 / 52 + 40 us; the stage by the columns too, 51 + 27 / 54 + 38,
// leaves less to share between the blocks of a tile: 1500 tokens 69 + 49 and 67 + 45).
// All of it together, us before and now of the best tile for routings by chance: 400 / 800 / 1100 / 1500 / 2048 / 2500 / 3000 / 4000 / 8000 tokens 98 / 107 / 119 / 125 /
// 173 / 187 / 192 / 270 / 450 -> 75 / 93 / 114 / 115 / 143 / 181 / 192 / 236 / 420.  Before that loop, by the kernel above, gate|up took
// 160 us at 2048 tokens and 470 at 8192.  Blocks of 128 x 128 or 128 x 256 with one barrier and all reads of a stage ahead of its products
// took 127 to 150 us at 2048 tokens, whatever the number of stages; a wave of its own that asked for the matrix's lines ahead
// of time made them slower (180 us).
template <class T, bool GATED>
__device__ __forceinline__ void moe_products_tile(unsigned char* stages, const bf16_t* __restrict__ x, int ldx, const int* __restrict__ row_index,
                                                  const bf16_t* __restrict__ w, int e, int slot0, int rows, int n0,
                                                  void* __restrict__ out_, int ldo, int n_out, int K, float limit, float alpha) {
  constexpr int COLS = GATED ? 128 : 256;                // output columns of a block
  constexpr int H = T::STRIP, WN = 8 / H;                // 16-row pieces of a wave's strip of W, waves beside each other
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const size_t w_rows = GATED ? 2 * (size_t)n_out : (size_t)n_out;
  unsigned xoff[T::XL], woff[T::WL];
#pragma unroll
  for (int i = 0; i < T::XL; ++i) {
    const int row = T::x_row(wave, lane, i), slot = slot0 + (row < rows ? row : rows - 1);
    xoff[i] = 2u * ((unsigned)(row_index ? row_index[slot] : slot) * (unsigned)ldx + T::k_of(row, lane));
  }
#pragma unroll
  for (int i = 0; i < T::WL; ++i) {
    const int row = T::w_row(wave, lane, i);
    int n = n0 + row % COLS;
    if (n >= n_out) n = n_out - 1;
    woff[i] = 2u * ((unsigned)((GATED && row >= COLS ? n_out : 0) + n) * (unsigned)K + T::k_of(row, lane));
  }
  tile_f32x4 acc[T::TN][T::TM];
  T::run(stages, reinterpret_cast<const char*>(x), xoff, reinterpret_cast<const char*>(w + (size_t)e * w_rows * K), woff,
         K >> 6, T::TURNED ? (int)((unsigned)e % (unsigned)(K >> 6)) : 0, wave, lane, 128, acc);
  // lane (r, g): row r of each 16-row group, four consecutive columns at 4g
  const int wm = wave / WN, wn = wave % WN;
  const bool whole = ((n_out | ldo) & (GATED ? 7 : 3)) == 0 && !((uintptr_t)out_ & 15);
#pragma unroll
  for (int m = 0; m < T::TM; ++m) {
    const int row = 64 * wm + 16 * m + r;
    if (row >= rows) continue;
    if (whole) {
      if constexpr (!GATED) {
        float* const o = reinterpret_cast<float*>(out_) + (size_t)(slot0 + row) * ldo;
#pragma unroll
        for (int n = 0; n < 2 * H; ++n) {
          const int c = n0 + 16 * H * wn + 16 * (n % H) + 4 * g + (n < H ? 0 : 128);
          if (c < n_out) *reinterpret_cast<float4*>(o + c) = make_float4(acc[n][m][0], acc[n][m][1], acc[n][m][2], acc[n][m][3]);
        }
        continue;
      } else if constexpr (H > 1) {
#pragma unroll
        for (int n = 0; n < H; n += 2) {
          uint2 u[2];
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            float v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = moe_glu<false>(acc[n + h][m][i], acc[n + h + H][m][i], limit, alpha);
            u[h] = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
          }
          const uint4 both = pair_columns(u[0], u[1]);
          const int c = n0 + 16 * H * wn + 16 * n + pair_column(g);
          if (c < n_out) *reinterpret_cast<uint4*>(reinterpret_cast<bf16_t*>(out_) + (size_t)(slot0 + row) * ldo + c) = both;
        }
        continue;
      }
    }
#pragma unroll
    for (int n = 0; n < (GATED ? H : 2 * H); ++n) {
      const int c = n0 + 16 * H * wn + 16 * (n % H) + 4 * g + (n < H ? 0 : 128);
      const size_t at = (size_t)(slot0 + row) * ldo + c;
      if constexpr (GATED) {
        bf16_t* const o = reinterpret_cast<bf16_t*>(out_) + at;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = moe_glu<false>(acc[n][m][i], acc[n + H][m][i], limit, alpha);
        if (c + 3 < n_out && (ldo & 3) == 0) {
          *reinterpret_cast<uint2*>(o) = make_uint2(pack2_bf16(v[0], v[1]), pack2_bf16(v[2], v[3]));
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (c + i < n_out) o[i] = f32_to_bf16_bits(v[i]);
        }
      } else {
        float* const o = reinterpret_cast<float*>(out_) + at;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (c + i < n_out) o[i] = acc[n][m][i];
      }
    }
  }
}

// The tile and the block of its columns that this block takes, or a tile of -1: die d (blocks go to the dies round-robin) takes the
// d-th eighth of the tiles in use, a tile's columns side by side.
__device__ __forceinline__ int tile_in_turn(const int* __restrict__ tiles, int n_tiles, int n_col_blocks, int* columns) {
  const int total = tiles[3 * n_tiles] * n_col_blocks, per_die = (total + 7) / 8;
  const int item = ((int)blockIdx.x & 7) * per_die + ((int)blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_die || item >= total) return -1;
  *columns = item % n_col_blocks;
  return item / n_col_blocks;
}
// As above where the blocks fill whole rounds of a die's 32 units, or nearly, or where most experts have a tile of 64 rows or less:
// a tile's neighbours of the same expert then run beside it and share its matrix.  Else every die takes its eighth of the tiles of more than
// 64 rows, and behind them its eighth of the others, which take about half a round (32 experts of 256 rows by chance, half of them
// with a few rows more, gate|up 111 us in turn, 92 so; of 500 162 and 141, of 750 210 and 192; of 312, every one with a second tile, 104 in
// turn, 115 so; of 625 168 and 178).
__device__ __forceinline__ int tile_by_rows(const int* __restrict__ tiles, int n_tiles, int n_col_blocks, int* columns) {
  constexpr int HELD = 4;                                // 64 tiles each; a longer list makes many rounds
  const int lane = threadIdx.x & 63, die = (int)blockIdx.x & 7;
  int rows[HELD], big = 0;
#pragma unroll
  for (int i = 0; i < HELD; ++i) rows[i] = tiles[3 * (64 * i + lane < n_tiles ? 64 * i + lane : 0) + 2];   // beside the list's length
  const int used = tiles[3 * n_tiles], last = used * n_col_blocks & 255;
#pragma unroll
  for (int i = 0; i < HELD; ++i) {
    rows[i] = 64 * i + lane < used ? rows[i] : 0;
    big += __popcll(__ballot(rows[i] > 64));
  }
  if (used > 64 * HELD || used * n_col_blocks <= 256 || last == 0 || last > 204 || (used - big) * n_col_blocks > 160)
    return tile_in_turn(tiles, n_tiles, n_col_blocks, columns);
  int at = (int)blockIdx.x >> 3;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    unsigned long long of[HELD];
    int total = 0;
#pragma unroll
    for (int i = 0; i < HELD; ++i) {
      of[i] = __ballot(k == 0 ? rows[i] > 64 : rows[i] > 0 && rows[i] <= 64);
      total += n_col_blocks * __popcll(of[i]);
    }
    const int per_die = (total + 7) / 8, left = total - die * per_die, mine = left < per_die ? left : per_die;
    if (at < mine) {
      const int item = die * per_die + at;
      int nth = item / n_col_blocks;
      *columns = item % n_col_blocks;
#pragma unroll
      for (int i = 0; i < HELD; ++i) {
        const int here = __popcll(of[i]);
        if (nth < here) return 64 * i + __ffsll(__ballot((of[i] >> lane & 1) && __popcll(of[i] & ((1ull << lane) - 1)) == nth)) - 1;
        nth -= here;
      }
    }
    at -= mine > 0 ? mine : 0;
  }
  return -1;
}

template <int WMW, int STAGES, bool GATED, bool TURNED>
__global__ void __launch_bounds__(128 * WMW)
moe_products_kernel(const bf16_t* __restrict__ x, int ldx, const int* __restrict__ row_index,
                    const bf16_t* __restrict__ w, const int* __restrict__ tiles, int n_tiles, int n_col_blocks,
                    void* __restrict__ out, int ldo, int n_out, int K, float limit, float alpha) {
  extern __shared__ __attribute__((aligned(16))) unsigned char tile_stages[];
  int item;
  const int tile = WMW == 4 ? tile_by_rows(tiles, n_tiles, n_col_blocks, &item) : tile_in_turn(tiles, n_tiles, n_col_blocks, &item);
  if (tile < 0) return;
  const int n0 = item * (GATED ? 128 : 256);
  const int e = tiles[3 * tile], slot0 = tiles[3 * tile + 1], rows = tiles[3 * tile + 2];
  if (rows <= 0) return;
#define TILE(...) moe_products_tile<__VA_ARGS__, GATED>(tile_stages, x, ldx, row_index, w, e, slot0, rows, n0, out, ldo, n_out, K, limit, alpha)
  if constexpr (WMW == 4) {
    if (rows <= 64) return TILE(ProductTiles<1, 3, 8, TURNED>);
  }
  TILE(ProductTiles<WMW, STAGES, 2, TURNED>);
#undef TILE
}

// Rows of a tile the matrix-core kernels take for a launch made with `tile_rows` rows a tile.
extern "C" int ullm_moe_mfma_supports(int K, int ldx, int tile_rows) {
  return K >= 8 && K % 8 == 0 && ldx % 8 == 0 && (tile_rows == 16 || tile_rows == 32 || tile_rows == 64 || tile_rows == 128 ||
                                                  (tile_rows == 256 && K % 64 == 0));
}

template <int MT, bool GATED, typename... Args>
static void launch_tiles(dim3 grid, hipStream_t stream, Args... args) {
  constexpr int bytes = 2 * (16 * MT * 128 + 128 * 128);
  static const hipError_t allowed = hipFuncSetAttribute((const void*)moe_tiles_mfma_kernel<MT, GATED>,
                                                        hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  (void)allowed;
  hipLaunchKernelGGL((moe_tiles_mfma_kernel<MT, GATED>), grid, dim3(256), bytes, stream, args...);
}

template <int MT, bool GATED, typename... Args>
static void launch_rows_dma(dim3 grid, hipStream_t stream, Args... args) {
  constexpr int bytes = 4 * 2 * ((GATED ? 32 : 16) + 16 * MT) * 128;          // 32, 48 or 64 KB
  hipLaunchKernelGGL((moe_rows_dma_kernel<MT, GATED>), grid, dim3(256), bytes, stream, args...);
}

// Experts begin K at different stages from this K on, whatever the tile (a row's sums do not depend on the rows beside it): us of gate|up + down from one stage and so, 32 experts, width 2048, 1024 columns
// 24 / 80 / 220 rows an expert 98 / 108 / 143 and 80 / 87 / 134, 16 experts of them 56 / 64 / 71 and 51 / 60 / 67; with both products' rows shorter
// they were slower so (64 experts, width 1024, 768 columns 71 / 82 / 139 and 75 / 84 / 145, 40 experts, width 1536 93 / 102 / 145 and 96 / 106 / 148).
#define TURNED_K 2048
template <int WMW, int STAGES, bool GATED, bool TURNED, typename... Args>
static void launch_products(dim3 grid, hipStream_t stream, Args... args) {
  constexpr int bytes = ProductTiles<WMW, STAGES>::BYTES;
  static_assert(WMW != 4 || bytes >= ProductTiles<1, 3, 8>::BYTES, "the largest of a launch's");
  static const hipError_t allowed = hipFuncSetAttribute((const void*)moe_products_kernel<WMW, STAGES, GATED, TURNED>,
                                                        hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  (void)allowed;
  hipLaunchKernelGGL((moe_products_kernel<WMW, STAGES, GATED, TURNED>), grid, dim3(128 * WMW), bytes, stream, args...);
}

// out[slot] = glu(x[row_index[slot]] Wg^T, x Wu^T) (gated: out in x's dtype, w [experts, 2 n_out, K]) or
// x[slot] W^T (not gated: out float32, w [experts, n_out, K]) over the tiles' rows.  row_index may be null.
extern "C" int ullm_moe_rows(const void* x, int ldx, const int* row_index, const void* w, const int* tiles,
                             int max_tiles, int tile_rows, void* out, int ldo, int n_out, int K, int gated,
                             float limit, float alpha, int dtype, hipStream_t stream) {
  if (max_tiles <= 0) return 0;
  if (n_out < 1 || K < 1 || ldx < K || ldo < n_out || tile_rows < 1) return ULLM_ERR_SHAPE;
  if (dtype == ULLM_BF16 && ullm_moe_mfma_supports(K, ldx, tile_rows) && !((uintptr_t)x & 15) && !((uintptr_t)w & 15)) {
    // the loop's loads count bytes from x and from the expert's matrix in 32 bits (a row of x is a token or a slot: never past
    // the slots of all tiles)
    const bool near = (long long)max_tiles * tile_rows * ldx < (1LL << 31) && (gated ? 2LL : 1LL) * n_out * K < (1LL << 31);
    if (tile_rows >= 128 && K % 64 == 0 && near) {
      const int per_block = gated ? 128 : 256, col_blocks = (n_out + per_block - 1) / per_block;
      const long long total = (long long)max_tiles * col_blocks;
      if (total > 0x3fffffffLL) return ULLM_ERR_SHAPE;
      dim3 grid((unsigned)(8 * ((total + 7) / 8 + (tile_rows == 256 ? 1 : 0))));   // two eighths, each rounded up
#define TILES(W, ST, G, TURNED) launch_products<W, ST, G, TURNED>(grid, stream, (const bf16_t*)x, ldx, row_index, (const bf16_t*)w, tiles, max_tiles, \
    col_blocks, out, ldo, n_out, K, limit, alpha)
#define TILES_BY(TURNED) do {                                                                                   \
        if (tile_rows == 256) { if (gated) TILES(4, 2, true, TURNED); else TILES(4, 2, false, TURNED); }         \
        else { if (gated) TILES(2, 3, true, TURNED); else TILES(2, 3, false, TURNED); }                          \
      } while (0)
      if (K >= TURNED_K) TILES_BY(true);
      else TILES_BY(false);
#undef TILES_BY
#undef TILES
      ULLM_LAUNCH_CHECK();
    }
    if (tile_rows == 256) return ULLM_ERR_SHAPE;
    if (tile_rows >= 64) {
      const int col_blocks = (n_out + (gated ? 63 : 127)) / (gated ? 64 : 128);
      const long long total = (long long)max_tiles * col_blocks;
      if (total > 0x3fffffffLL) return ULLM_ERR_SHAPE;
      dim3 grid((unsigned)(8 * ((total + 7) / 8)));
#define TILES(MT, G) launch_tiles<MT, G>(grid, stream, (const bf16_t*)x, ldx, row_index, (const bf16_t*)w, tiles, max_tiles, \
    col_blocks, out, ldo, n_out, K, limit, alpha)
      if (tile_rows == 64) { if (gated) TILES(4, true); else TILES(4, false); }
      else { if (gated) TILES(8, true); else TILES(8, false); }
#undef TILES
      ULLM_LAUNCH_CHECK();
    }
    dim3 grid(max_tiles, (n_out + 15) / 16), block(256);
    if (grid.y > 65535) return ULLM_ERR_SHAPE;
    if (K % 64 == 0 && K >= 256) {
#define GO(MT, G) launch_rows_dma<MT, G>(grid, stream, (const bf16_t*)x, ldx, row_index, (const bf16_t*)w, tiles, out, ldo, n_out, K, limit, alpha)
      if (tile_rows == 16) { if (gated) GO(1, true); else GO(1, false); }
      else { if (gated) GO(2, true); else GO(2, false); }
#undef GO
      ULLM_LAUNCH_CHECK();
    }
#define GO(MT, G) hipLaunchKernelGGL((moe_rows_mfma_kernel<MT, G>), grid, block, 0, stream, (const bf16_t*)x, ldx, row_index, \
    (const bf16_t*)w, tiles, out, ldo, n_out, K, limit, alpha)
    if (tile_rows == 16) { if (gated) GO(1, true); else GO(1, false); }
    else { if (gated) GO(2, true); else GO(2, false); }
#undef GO
    ULLM_LAUNCH_CHECK();
  }
  if ((size_t)K * sizeof(float) > 64 * 1024) return ULLM_ERR_SHAPE;
  const int cols_per_block = 64;
  dim3 grid(max_tiles, (n_out + cols_per_block - 1) / cols_per_block), block(256);
  if (grid.y > 65535) return ULLM_ERR_SHAPE;
  const size_t lds = (size_t)K * sizeof(float);
#define GO(TT, G) hipLaunchKernelGGL((moe_rows_simple_kernel<TT, G>), grid, block, lds, stream, (const TT*)x, ldx, row_index, \
    (const TT*)w, tiles, out, ldo, n_out, K, cols_per_block, limit, alpha)
  if (dtype == ULLM_F32) { if (gated) GO(float, true); else GO(float, false); }
  else if (dtype == ULLM_BF16) { if (gated) GO(bf16_t, true); else GO(bf16_t, false); }
  else return ULLM_ERR_DTYPE;
#undef GO
  ULLM_LAUNCH_CHECK();
}

// ------------------------------------------------------------------------------- the weighted sum
// out[t][c] = base[t][c] + bias[c] + shared[t][c] + sum_k weights[t][k] * (ids[t][k] < n_experts ? y[slot][c] : x[t][c]);
// base (float32 or TX), bias (float32), shared (TX) may be null.  grid (tokens, groups of columns): a thread takes
// VEC consecutive columns, all its loads independent of each other.
//
// TANH: on its way into the stream and through the squashing that the next sublayers read, which looks at no other column:
// residual += mult * sum, squashed = tanh(alpha * residual) * gain + shift, as elementwise.hip's add_tanh_kernel does from a sum in memory.
// What bounds it is bytes: without it the sum was written and read again by a launch of its own.  4 of 32 experts of width 2048, us for both
// launches -> this one: 1 token 5.7 -> 4.3, 48 6.3 -> 4.4, 300 8.5 -> 5.5, 1000 18.5 -> 14.2, 3000 41.5 -> 33.8.
// (One kernel with the sum in its body and its pointers one by one.  As a function of a structure's pointers, which may point anywhere, loads wait for each
// other: 3000 tokens, 4 of width 2048, with a base and a shared expert 29.4 us and so 27.0, 48 tokens 3.86 and 3.64.)
template <typename TX, typename TB, int VEC, bool TANH>
__global__ void __launch_bounds__(256)
moe_combine_kernel(const float* __restrict__ y, const TX* __restrict__ x, int ldx, const int* __restrict__ ids,
                   const float* __restrict__ weights, const int* __restrict__ slot_of_pair, int top, int n_experts,
                   const TB* __restrict__ base, const float* __restrict__ bias, const TX* __restrict__ shared,
                   float* __restrict__ out, int H, float mult, float* __restrict__ residual, const float* __restrict__ alpha,
                   const float* __restrict__ gain, const float* __restrict__ shift, TX* __restrict__ squashed) {
  const int t = blockIdx.x, c = VEC * (blockIdx.y * 256 + threadIdx.x);
  if (c >= H) return;
  float r[VEC], g[VEC], h[VEC], by = 0.f;
  if constexpr (TANH) {
    by = *alpha;
#pragma unroll
    for (int i = 0; i < VEC; ++i) r[i] = residual[(size_t)t * H + c + i], g[i] = gain[c + i], h[i] = shift[c + i];
  }
  float a[VEC];
#pragma unroll
  for (int i = 0; i < VEC; ++i) {
    a[i] = base ? ld_f32(base + (size_t)t * H + c + i) : 0.f;
    if (bias) a[i] += bias[c + i];
    if (shared) a[i] += ld_f32(shared + (size_t)t * H + c + i);
  }
  for (int k = 0; k < top; ++k) {
    const int e = ids[(size_t)t * top + k];
    const float wk = weights[(size_t)t * top + k];
    if (e < n_experts) {
      const float* yr = y + (size_t)slot_of_pair[(size_t)t * top + k] * H + c;
#pragma unroll
      for (int i = 0; i < VEC; ++i) a[i] = fmaf(wk, yr[i], a[i]);
    } else {
#pragma unroll
      for (int i = 0; i < VEC; ++i) a[i] = fmaf(wk, ld_f32(x + (size_t)t * ldx + c + i), a[i]);
    }
  }
#pragma unroll
  for (int i = 0; i < VEC; ++i) {
    if constexpr (TANH) {
      r[i] += mult * a[i];
      residual[(size_t)t * H + c + i] = r[i];
      st_f32(squashed + (size_t)t * H + c + i, tanhf(by * r[i]) * g[i] + h[i]);
    } else {
      out[(size_t)t * H + c + i] = a[i];
    }
  }
}

// What both sums look at before a launch.
static int bad_combine(int top, int ldx, int T_, int H, const void* base, int base_dtype, int dtype) {
  if (H < 1 || top < 1 || ldx < H || (H / (H % 4 == 0 ? 4 : 1) + 255) / 256 > 65535) return ULLM_ERR_SHAPE;
  if (dtype != ULLM_F32 && dtype != ULLM_BF16) return ULLM_ERR_DTYPE;
  return base && dtype == ULLM_F32 && base_dtype != ULLM_F32 ? ULLM_ERR_DTYPE : 0;
}
// Calls GO(TX, TB, VEC) for the rows' type, the base's and how many columns a thread takes.
#define COMBINE_BY_TYPES() do { \
    if (dtype == ULLM_F32) { if (vec == 4) GO(float, float, 4); else GO(float, float, 1); } \
    else if (base && base_dtype == ULLM_BF16) { if (vec == 4) GO(bf16_t, bf16_t, 4); else GO(bf16_t, bf16_t, 1); } \
    else { if (vec == 4) GO(bf16_t, float, 4); else GO(bf16_t, float, 1); } } while (0)
#define COMBINE_ARGS(TX, TB) y, (const TX*)x, ldx, ids, weights, slot_of_pair, top, n_experts, (const TB*)base, bias, (const TX*)shared

extern "C" int ullm_moe_combine(const float* y, const void* x, int ldx, const int* ids, const float* weights,
                                const int* slot_of_pair, int top, int n_experts, const void* base, int base_dtype,
                                const float* bias, const void* shared, float* out, int T_, int H, int dtype,
                                hipStream_t stream) {
  if (T_ <= 0) return 0;
  if (const int bad = bad_combine(top, ldx, T_, H, base, base_dtype, dtype)) return bad;
  const int vec = H % 4 == 0 ? 4 : 1;
  dim3 grid(T_, (H / vec + 255) / 256), block(256);
#define GO(TX, TB, V) hipLaunchKernelGGL((moe_combine_kernel<TX, TB, V, false>), grid, block, 0, stream, COMBINE_ARGS(TX, TB), out, H, \
    0.f, (float*)nullptr, (const float*)nullptr, (const float*)nullptr, (const float*)nullptr, (TX*)nullptr)
  COMBINE_BY_TYPES();
#undef GO
  ULLM_LAUNCH_CHECK();
}

// out [T, H] of the rows' type
extern "C" int ullm_moe_combine_tanh(const float* y, const void* x, int ldx, const int* ids, const float* weights,
                                     const int* slot_of_pair, int top, int n_experts, const void* base, int base_dtype,
                                     const float* bias, const void* shared, float mult, float* residual, const float* alpha, const float* gain,
                                     const float* shift, void* out, int T_, int H, int dtype, hipStream_t stream) {
  if (T_ <= 0) return 0;
  if (const int bad = bad_combine(top, ldx, T_, H, base, base_dtype, dtype)) return bad;
  const int vec = H % 4 == 0 ? 4 : 1;
  dim3 grid(T_, (H / vec + 255) / 256), block(256);
#define GO(TX, TB, V) hipLaunchKernelGGL((moe_combine_kernel<TX, TB, V, true>), grid, block, 0, stream, COMBINE_ARGS(TX, TB), (float*)nullptr, H, \
    mult, residual, alpha, gain, shift, (TX*)out)
  COMBINE_BY_TYPES();
#undef GO
  ULLM_LAUNCH_CHECK();
}
#undef COMBINE_ARGS
#undef COMBINE_BY_TYPES
