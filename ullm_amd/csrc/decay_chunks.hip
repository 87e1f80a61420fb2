// The recurrence of decay_scan.hip for long portions of prompts, in chunks of 16 tokens on the 32-bit matrix cores and in
// segments of chunks that are worked side by side.
//
// Inside a chunk, with S0 the state it finds, G_ij[n] = d_(j+1)[n] .. d_i[n], c_i = G_i0 and C = c_16:
//   o_i = (q_i c_i)^T S0 + sum_(j<=i) A_ij v_j,   A_ij = sum_n q_i[n] G_ij[n] k_j[n]
//   S1 = diag(C) S0 + sum_j (k_j G_16,j) v_j^T
// (outputs before the update: c and G run to i - 1, and A_ii = sum_n q_i[n] u[n] k_i[n].)  Three passes and a fourth where a
// request has several segments:
//   chunk      for every chunk and head q_i c_i, k_j G_16,j (turned, tokens side by side), C and A, all chunks at once
//   segment    the state every segment but a request's last would leave if it began with zeros, and its decays' product
//   carry      the states the segments find, one after the other (a multiply-add per segment and element)
//   out        outputs, and the last segment's state
// Decays' products are formed as products: no logarithm, no quotient.  Everything is 32-bit.
//
// What bounds it: the walk over a request's tokens one by one was a chain of 2048 steps in 256 blocks.  Here a wave has 68
// products of 32 cycles a chunk, and sixteen segments fill the chip.  2048 tokens,
// 16 heads of 128 x 128, decays per head / per channel: 295 / 308 us token by token, 100 / 109 us here; 3000 tokens of four
// requests 214 / 209 and 134 / 149 us.
#include "common.h"
#include "decay_inputs.h"

typedef __attribute__((ext_vector_type(4))) float f32x4_t;
#define CHUNK 16

// D[i][j] += sum_k A[i][k] B[k][j], 16 x 4 by 4 x 16: lane (c, g) = (lane % 16, lane / 16) holds A[c][k], B[k][c] for its own k and
// D[4 g + r][c] in register r.  Which k a lane group stands for is free as long as A and B agree: a 16 x 16 result's register r
// is, as it lies, the B operand of the step whose groups stand for k = 4 g + r.
__device__ __forceinline__ f32x4_t mma(float a, float b, f32x4_t c) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
#else
  return c;
#endif
}

struct ChunkArgs {
  const float* q;
  const float* k;
  const float* v;
  const float* z;             // raw decays [T, heads * N] or the heads' constants
  const float* bonus;         // [heads, N]: outputs before the update; or null
  float* state;
  long long state_stride, state_off;
  const int* entry_slot;
  const int* items;           // per chunk (first token, tokens)
  const int* segments;        // per segment (entry, first chunk, chunks, its number in the entry, segments of the entry)
  const int* entry_segment;   // [entries]: an entry's first segment
  float* chunks;              // [chunks, heads, 33 N + 256]
  float* carried;             // [segments, heads, N P + N]: states (first those the segments leave, then those they find), decays
  float* out;                 // [T, heads * P]
  int q_ld, k_ld, v_ld, z_ld;
  int heads, N, P, decay_kind, silu_inputs, write_state;
  float q_scale, inv_tau;
};
// a chunk and head's part of `chunks`: q_i c_i [16][N], k_j G_16,j [N][16], A [16][16], C [N]
__device__ __forceinline__ size_t chunk_floats(int N) { return 33 * (size_t)N + 256; }

// One wave per (chunk, head), the lanes side by side along the key channels, 64 at a time.
__global__ void __launch_bounds__(64)
decay_chunk_kernel(const ChunkArgs a) {
  const int item = blockIdx.x, h = blockIdx.y, lane = threadIdx.x, N = a.N;
  const int t0 = a.items[2 * item], n_tok = a.items[2 * item + 1];
  float* to = a.chunks + ((size_t)item * a.heads + h) * chunk_floats(N);
  const bool before = a.bonus != nullptr;
  float pair[128], same[CHUNK];                          // A_ij (j < i) at i (i - 1) / 2 + j, and A_ii
#pragma unroll
  for (int p = 0; p < 128; ++p) pair[p] = 0.f;
#pragma unroll
  for (int i = 0; i < CHUNK; ++i) same[i] = 0.f;
  for (int n0 = 0; n0 < N; n0 += 64) {
    const int n = n0 + lane, at = n < N ? n : N - 1;
    float q[CHUNK], k[CHUNK], d[CHUNK];
#pragma unroll
    for (int i = 0; i < CHUNK; ++i) {
      const size_t t = t0 + (i < n_tok ? i : n_tok - 1);
      q[i] = a.q[t * a.q_ld + (size_t)h * N + at];
      k[i] = a.k[t * a.k_ld + (size_t)h * N + at];
      d[i] = a.decay_kind == DECAY_PER_HEAD ? a.z[h] : a.z[t * a.z_ld + (size_t)h * N + at];
    }
    const float u = before ? a.bonus[(size_t)h * N + at] : 1.f;
#pragma unroll
    for (int i = 0; i < CHUNK; ++i) {
      if (a.silu_inputs) q[i] = exact_silu(q[i]), k[i] = exact_silu(k[i]);
      q[i] *= a.q_scale;
      if (a.decay_kind == DECAY_SIGMOID_ROOT || a.decay_kind == DECAY_EXP_EXP) d[i] = decay_of(d[i], a.decay_kind, a.inv_tau);
      if (i >= n_tok || n >= N) q[i] = 0.f, k[i] = 0.f, d[i] = 1.f;      // nothing read, nothing taken, nothing lost
    }
    float c = 1.f;
#pragma unroll
    for (int i = 0; i < CHUNK; ++i) {
      const float after = c * d[i];
      if (n < N) to[(size_t)i * N + n] = q[i] * (before ? c : after);
      c = after;
    }
    if (n < N) to[32 * (size_t)N + 256 + n] = c;
    float kt[CHUNK];
    c = 1.f;
#pragma unroll
    for (int j = CHUNK - 1; j >= 0; --j) {
      kt[j] = k[j] * c;
      c *= d[j];
    }
    if (n < N) {
#pragma unroll
      for (int j = 0; j < CHUNK; j += 4)
        *reinterpret_cast<float4*>(to + 16 * (size_t)N + 16 * (size_t)n + j) = make_float4(kt[j], kt[j + 1], kt[j + 2], kt[j + 3]);
    }
#pragma unroll
    for (int j = 0; j < CHUNK; ++j) {
      same[j] = fmaf(q[j], u * k[j], same[j]);
      float w = k[j];
#pragma unroll
      for (int i = j + 1; i < CHUNK; ++i) {
        if (!before) w *= d[i];
        pair[i * (i - 1) / 2 + j] = fmaf(q[i], w, pair[i * (i - 1) / 2 + j]);
        if (before) w *= d[i];
      }
    }
  }
  // the lanes' sums: at every step a lane gives half of its values away and adds up the other half; lane l ends with
  // values 2 l and 2 l + 1
#pragma unroll
  for (int s = 0; s < 6; ++s) {
    const int half = 64 >> s, mask = 32 >> s;
    const bool upper = lane & mask;
#pragma unroll
    for (int p = 0; p < half; ++p) {
      const float keep = upper ? pair[p + half] : pair[p], give = upper ? pair[p] : pair[p + half];
      pair[p] = keep + __shfl_xor(give, mask, 64);
    }
  }
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const int half = 8 >> s, mask = 32 >> s;
    const bool upper = lane & mask;
#pragma unroll
    for (int p = 0; p < half; ++p) {
      const float keep = upper ? same[p + half] : same[p], give = upper ? same[p] : same[p + half];
      same[p] = keep + __shfl_xor(give, mask, 64);
    }
  }
  same[0] += __shfl_xor(same[0], 2, 64);
  same[0] += __shfl_xor(same[0], 1, 64);
  float* const A = to + 32 * (size_t)N;
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int p = 2 * lane + e;
    int i = 1;
    while (i * (i + 1) / 2 <= p) ++i;
    if (p < 120) A[16 * i + p - i * (i - 1) / 2] = pair[e];
  }
  if ((lane & 3) == 0) A[17 * (lane >> 2)] = same[0];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int i = lane >> 2, j = 4 * (lane & 3) + e;
    if (j > i) A[16 * i + j] = 0.f;
  }
}

// The values of v at this lane's column for tokens 4 g .. 4 g + 3 of a chunk; past the portion's end nothing.
__device__ __forceinline__ f32x4_t chunk_values(const ChunkArgs& a, int t0, int n_tok, int h, int col, int g) {
  f32x4_t v;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = 4 * g + r;
    v[r] = a.v[(size_t)(t0 + (i < n_tok ? i : n_tok - 1)) * a.v_ld + (size_t)h * a.P + col];
  }
  return v;
}
__device__ __forceinline__ void finish_values(const ChunkArgs& a, int n_tok, int g, f32x4_t& v) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    if (a.silu_inputs) v[r] = exact_silu(v[r]);
    if (4 * g + r >= n_tok) v[r] = 0.f;
  }
}

// A wave takes 16 value columns of a head and keeps the state's NT row tiles of them in registers over the chunks of a
// segment; nothing passes between waves.  OUT: outputs too (a chunk's reads of the state before its update); else only the
// state, from zeros, and the decays' product.  What the next chunk needs is asked for as soon as this one's is used up.
template <int NT, bool OUT>
__global__ void __launch_bounds__(512)
decay_segment_kernel(const ChunkArgs a) {
  const int seg = blockIdx.x, h = blockIdx.y;
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tile = blockIdx.z * (blockDim.x >> 6) + wave, N = a.N, P = a.P, col = 16 * tile + c;
  const int* s_at = a.segments + 5 * seg;
  const int entry = s_at[0], first = s_at[1], n_chunks = s_at[2], number = s_at[3], of = s_at[4];
  if (16 * tile >= P || (!OUT && number + 1 == of)) return;
  float* const row = a.state + (size_t)a.entry_slot[entry] * a.state_stride + a.state_off + (size_t)h * N * P + col;
  float* const carried = a.carried + ((size_t)seg * a.heads + h) * ((size_t)N * P + N);
  f32x4_t S[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      S[t][r] = !OUT ? 0.f : (of > 1 ? carried + col : row)[(size_t)(16 * t + 4 * g + r) * P];
  f32x4_t q[NT], k[NT], keep[NT], tri, v, all[OUT ? 1 : NT];
  if constexpr (!OUT) {
#pragma unroll
    for (int t = 0; t < NT; ++t) all[t] = f32x4_t{1.f, 1.f, 1.f, 1.f};
  }
  const size_t step = a.heads * chunk_floats(N);
  const float* at = a.chunks + ((size_t)first * a.heads + h) * chunk_floats(N);
  auto fetch_q = [&](const float* p) __attribute__((always_inline)) {
    if constexpr (OUT) {
#pragma unroll
      for (int t = 0; t < NT; ++t) q[t] = *reinterpret_cast<const f32x4_t*>(p + (size_t)c * N + 16 * t + 4 * g);
      tri = *reinterpret_cast<const f32x4_t*>(p + 32 * (size_t)N + 16 * c + 4 * g);
    }
  };
  auto fetch_k = [&](const float* p) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < NT; ++t) k[t] = *reinterpret_cast<const f32x4_t*>(p + 16 * (size_t)N + 16 * (size_t)(16 * t + c) + 4 * g);
#pragma unroll
    for (int t = 0; t < NT; ++t) keep[t] = *reinterpret_cast<const f32x4_t*>(p + 32 * (size_t)N + 256 + 16 * t + 4 * g);
  };
  int t0 = a.items[2 * first], n_tok = a.items[2 * first + 1];
  fetch_q(at);
  fetch_k(at);
  v = chunk_values(a, t0, n_tok, h, col, g);
  for (int i = 0; i < n_chunks; ++i) {
    const int nx = first + (i + 1 < n_chunks ? i + 1 : i);             // behind the last chunk that one again
    const int t1 = a.items[2 * nx], n1 = a.items[2 * nx + 1];
    if (i + 1 < n_chunks) at += step;
    finish_values(a, n_tok, g, v);
    if constexpr (OUT) {
      f32x4_t o[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) o[r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = mma(q[t][r], S[t][r], o[r]);
      const bool fine = isfinite(v[0]) && isfinite(v[1]) && isfinite(v[2]) && isfinite(v[3]);
      if (__all(fine)) {
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = mma(tri[r], v[r], o[r]);
      } else {
        // a value that is not finite must not meet the zeros of earlier tokens' rows: token by token
        for (int j = 0; j < 16; ++j) {
          const int src = 16 * (j >> 2) + c, r = j & 3;
          const float vj = __shfl(r == 0 ? v[0] : r == 1 ? v[1] : r == 2 ? v[2] : v[3], src, 64);
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            const float mine = r == 0 ? tri[0] : r == 1 ? tri[1] : r == 2 ? tri[2] : tri[3];
            const float A = __shfl(mine, 16 * (j >> 2) + 4 * g + x, 64);          // A[4 g + x][j] lies in lane (4 g + x, j / 4)
            if (j <= 4 * g + x) o[0][x] += A * vj;
          }
        }
      }
      fetch_q(at);
      const f32x4_t sum = (o[0] + o[1]) + (o[2] + o[3]);
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (4 * g + r < n_tok) a.out[(size_t)(t0 + 4 * g + r) * a.heads * P + (size_t)h * P + col] = sum[r];
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      S[t] *= keep[t];
      if constexpr (!OUT) all[t] *= keep[t];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int t = 0; t < NT; ++t) S[t] = mma(k[t][r], v[r], S[t]);
    fetch_k(at);
    v = chunk_values(a, t1, n1, h, col, g);
    t0 = t1, n_tok = n1;
  }
  if (OUT ? !(a.write_state && number + 1 == of) : false) return;
  float* const to = OUT ? row : carried + col;
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) to[(size_t)(16 * t + 4 * g + r) * P] = S[t][r];
  if constexpr (!OUT) {
    if (tile == 0 && c == 0) {
#pragma unroll
      for (int t = 0; t < NT; ++t) *reinterpret_cast<f32x4_t*>(carried + (size_t)N * P + 16 * t + 4 * g) = all[t];
    }
  }
}

// A thread takes one element of a head's state through an entry's segments: what a segment leaves is replaced by what it
// finds.
__global__ void __launch_bounds__(256)
decay_carry_kernel(const ChunkArgs a) {
  const int entry = blockIdx.x, h = blockIdx.y, e = blockIdx.z * 256 + threadIdx.x;
  const int size = a.N * a.P;
  const int first = a.entry_segment[entry], of = a.segments[5 * first + 4];
  if (of == 1 || e >= size) return;
  float s = a.state[(size_t)a.entry_slot[entry] * a.state_stride + a.state_off + (size_t)h * size + e];
  const size_t step = a.heads * ((size_t)size + a.N);
  float* at = a.carried + ((size_t)first * a.heads + h) * ((size_t)size + a.N) + e;
  const int n = size + e / a.P - e;                       // from the element to its row's decay
  for (int i = 0; i < of; ++i, at += step) {
    if (i + 1 < of) {
      const float left = at[0], d = at[n];
      at[0] = s;
      s = d * s + left;
    } else {
      at[0] = s;
    }
  }
}

// key channels in whole tiles whose state fits a wave's registers beside its operands
extern "C" int ullm_decay_chunks_supports(int N, int P) {
  return (N == 16 || N == 32 || N == 48 || N == 64 || N == 80 || N == 96 || N == 128) && P >= 16 && P % 16 == 0 && P <= 65535;
}

extern "C" int ullm_decay_chunks(const float* q, int q_ld, const float* k, int k_ld, const float* v, int v_ld, const float* z, int z_ld,
                                 int decay_kind, float tau, const float* bonus, int silu_inputs, float q_scale, float* state,
                                 long long state_stride, long long state_off, const int* entry_slot, const int* items,
                                 int n_chunks, const int* segments, int n_segments, const int* entry_segment, int several,
                                 float* chunks, float* carried, float* out, int B_, int heads, int N, int P, int write_state,
                                 hipStream_t stream) {
  if (B_ <= 0 || n_chunks <= 0) return 0;
  if (heads <= 0 || heads > 65535 || n_segments <= 0 || !ullm_decay_chunks_supports(N, P)) return ULLM_ERR_SHAPE;
  if (decay_kind < DECAY_PER_HEAD || decay_kind > DECAY_READY || z == nullptr) return ULLM_ERR_UNSUPPORTED;
  if (decay_kind == DECAY_SIGMOID_ROOT && !(tau > 0.f)) return ULLM_ERR_UNSUPPORTED;
  ChunkArgs a;
  a.q = q, a.k = k, a.v = v, a.z = z, a.bonus = bonus, a.state = state, a.state_stride = state_stride, a.state_off = state_off;
  a.entry_slot = entry_slot, a.items = items, a.segments = segments, a.entry_segment = entry_segment, a.chunks = chunks;
  a.carried = carried, a.out = out, a.q_ld = q_ld, a.k_ld = k_ld, a.v_ld = v_ld, a.z_ld = z_ld, a.heads = heads, a.N = N, a.P = P;
  a.decay_kind = decay_kind, a.silu_inputs = silu_inputs, a.write_state = write_state, a.q_scale = q_scale;
  a.inv_tau = decay_kind == DECAY_SIGMOID_ROOT ? 1.f / tau : 1.f;
  hipLaunchKernelGGL(decay_chunk_kernel, dim3(n_chunks, heads), dim3(64), 0, stream, a);
  const int waves = P / 16 < 8 ? P / 16 : 8;
  const dim3 grid(n_segments, heads, (P / 16 + waves - 1) / waves), block(64 * waves);
  // NT row tiles: exactly N's
#define NT_GO(OUT) switch (N / 16) { \
    case 1: hipLaunchKernelGGL((decay_segment_kernel<1, OUT>), grid, block, 0, stream, a); break; \
    case 2: hipLaunchKernelGGL((decay_segment_kernel<2, OUT>), grid, block, 0, stream, a); break; \
    case 3: hipLaunchKernelGGL((decay_segment_kernel<3, OUT>), grid, block, 0, stream, a); break; \
    case 4: hipLaunchKernelGGL((decay_segment_kernel<4, OUT>), grid, block, 0, stream, a); break; \
    case 5: hipLaunchKernelGGL((decay_segment_kernel<5, OUT>), grid, block, 0, stream, a); break; \
    case 6: hipLaunchKernelGGL((decay_segment_kernel<6, OUT>), grid, block, 0, stream, a); break; \
    case 8: hipLaunchKernelGGL((decay_segment_kernel<8, OUT>), grid, block, 0, stream, a); break; \
    default: return ULLM_ERR_SHAPE; }
  if (several) {
    NT_GO(false);
    hipLaunchKernelGGL(decay_carry_kernel, dim3(B_, heads, (N * P + 255) / 256), dim3(256), 0, stream, a);
  }
  NT_GO(true);
#undef NT_GO
  ULLM_LAUNCH_CHECK();
}
