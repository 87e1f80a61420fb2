// What a block of prompt attention does with tiles that go straight to shared memory (attention_mfma.hip), as text: included in a
// function that several kernels call and, once more, in the kernel that is better off with it in its own body.  In scope: NQK, HEADS, KS,
// EXTRA, `block`, `lds`, `page_ids` and the kernel's arguments.
  using B = DmaBlock<NQK, HEADS, KS>;
  constexpr int TEAM = B::TEAM, SUBS = B::SUBS, TILES = B::TILES, TABLE = B::TABLE;
  using T = typename B::T;
  constexpr int HD = 32 * NQK;
  constexpr int NG = PREFILL_GROUPS;
  constexpr int PER_LANE = NG * (8 * NQK + 2);            // floats a lane hands over in the merge
  constexpr int PER = 2 * T::ROUNDS;                      // load instructions of a wave per tile
  static_assert((KS - 1) * TEAM * PER_LANE * 64 * 4 <= B::BYTES, "the merge reuses the tiles' memory");
  const int wave_id = (int)(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, wave = wave_id % TEAM, part = wave_id / TEAM;
  const int g = lane >> 4, c = lane & 15;
  unsigned char* const tile_lds = lds + part * TILES * T::BYTES;
  int* const pages = page_ids[part];
  const int G = nq / nkv, chunks = (G + HEADS - 1) / HEADS, per_kv = n_tiles * chunks;
  int kvh, rest;
  if (nkv % 8 == 0) {
    const int xcd = block & 7, slot = block >> 3;
    kvh = (slot / per_kv) * 8 + xcd;
    rest = slot % per_kv;
  } else {
    kvh = block / per_kv;
    rest = block % per_kv;
  }
  const int tile_idx = n_tiles - 1 - rest / chunks;
  const int head_in_group = (rest % chunks) * HEADS + wave % HEADS;
  const bool head_ok = head_in_group < G;                 // a wave without a head still helps to load
  const int head = kvh * G + (head_ok ? head_in_group : G - 1);
  extern __shared__ float dma_bias_stage[];
  const int bias_last = extras.bias_rows - 1;
  using BiasPtr = typename BiasPointer<EXTRA>::type;
  BiasPtr bias_row = nullptr;
  if constexpr (EXTRA) {
    if (extras.bias) {                                    // extras without a bias (a gate, a sink) stage nothing
      const float* const bias_global = extras.bias + (size_t)head * extras.bias_rows;
      for (int i = lane + 64 * part; i <= bias_last; i += 64 * KS) dma_bias_stage[wave * extras.bias_rows + i] = bias_global[i];
      bias_row = (lds_bias_ptr)dma_bias_stage + wave * extras.bias_rows;
    }
  }
  const int first = tiles[2 * tile_idx], count = tiles[2 * tile_idx + 1];
  // this wave's 32 tokens of the tile; a wave behind its end still helps to load
  const int skip = SUBS == 1 ? 0 : 16 * NG * (wave / HEADS);
  const int my_first = skip < count ? first + skip : first, my_count = count - skip < 16 * NG ? count - skip : 16 * NG;
  int clo[NG], chi[NG], tok[NG];
  Pack8 qreg[NG][NQK];
  const ScoreScale score_scale = split_scale(scale_log2e);
#pragma unroll
  for (int qg = 0; qg < NG; ++qg) {
    const bool ok = head_ok && 16 * qg + c < my_count;
    tok[qg] = my_first + (16 * qg + c < my_count ? 16 * qg + c : 0);
    const int pos = positions[tok[qg]];
    clo[qg] = first_seen_key(pos, window);
    chi[qg] = ok ? pos : -1;
    const bf16_t* qp = q + (size_t)tok[qg] * q_stride + (size_t)head * HD + 8 * g;
#pragma unroll
    for (int ch = 0; ch < NQK; ++ch) {
      if (ok) qreg[qg][ch].u4 = *reinterpret_cast<const uint4*>(qp + 32 * ch);
      else qreg[qg][ch].u4 = make_uint4(0, 0, 0, 0);
      // the power of two in scale * log2(e) goes into the queries once (exact); the scores take the rest
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const uint32_t two = qreg[qg][ch].w[w];
        qreg[qg][ch].w[w] = pack2_bf16(__uint_as_float(two << 16) * score_scale.pow2,
                                       __uint_as_float(two & 0xffff0000u) * score_scale.pow2);
      }
    }
  }
  const int last_pos = positions[first + count - 1];
  const int first_pos = positions[my_first];                // of this wave's tokens: what they see is open up to here
  const int open_lo = first_seen_key(last_pos, window);
  const int key_begin = first_seen_key(SUBS == 1 ? first_pos : positions[first], window) & ~31;
  const int key_end = last_pos + 1;
  const int steps = ((key_end - key_begin + 31) / 32 + KS - 1) / KS;    // this part's share of the 32-key tiles
  const int my_begin = key_begin + part * steps * 32;
  const int* bt = block_table + (size_t)token_entry[first] * bt_stride;
  f32x4_t acc[NG][2 * NQK];
  float m[NG], l[NG];
  f32x4_t negm[NG];
#pragma unroll
  for (int qg = 0; qg < NG; ++qg) {
#pragma unroll
    for (int n = 0; n < 2 * NQK; ++n) acc[qg][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    m[qg] = NEG_BIG;
    negm[qg] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    l[qg] = 0.f;
  }
  // where this lane reads its operands inside a tile: key row 8 (c / 4) + 4 sb + c % 4, piece 4 ch + g; dim 16 n + c, piece g
  int k_at[2][NQK];
#pragma unroll
  for (int sb = 0; sb < 2; ++sb)
#pragma unroll
    for (int ch = 0; ch < NQK; ++ch) {
      const int key = 8 * (c >> 2) + 4 * sb + (c & 3);
      k_at[sb][ch] = key * 2 * HD + 16 * ((4 * ch + g) ^ T::key_swizzle(key));
    }
  const int v_at = c * 64 + 16 * (g ^ (c >> 2));
  const DmaLanes<T> dl = dma_lanes<T>(page_size);
  const unsigned page_elems = (unsigned)(nkv * page_size * HD);
  const bf16_t* const k_head = k_pool + (size_t)kvh * page_size * HD;
  const bf16_t* const v_head = v_pool + (size_t)kvh * page_size * HD;
  // Tile i of this part is loaded with the page ids pages[2 (i - t0)], pages[2 (i - t0) + 1].
#define TILE_LOAD(I, T0) dma_tile_load<T>(tile_lds + ((I) % TILES) * T::BYTES, my_begin + 32 * (I), pages[2 * ((I) - (T0))], \
                                            pages[2 * ((I) - (T0)) + 1], page_size, dl, k_head, v_head, page_elems)
  // All tiles but one go on their way; in step i tile i + TILES - 1 follows, into the place of tile i - 1, which every wave
  // has left behind when it passes the step's barrier.  Loads are started for the tiles of this part's steps only,
  // so the last steps wait for fewer loads to be left.
  for (int t0 = 0; t0 < steps; t0 += DMA_TABLE_TILES) {
    // page ids of the tiles t0 .. t0 + DMA_TABLE_TILES + 3 (the loads run up to three tiles ahead of the steps)
    __syncthreads();
    for (int e = threadIdx.x & (64 * TEAM - 1); e < TABLE; e += 64 * TEAM) {
      const int kb = my_begin + 32 * t0 + 16 * e;
      pages[e] = kb < key_end ? bt[kb / page_size] : -1;
    }
    __syncthreads();
    if (t0 == 0) {
      if (steps > 0) TILE_LOAD(0, 0);
      if (TILES > 2 && steps > 1) TILE_LOAD(1, 0);
      if (TILES > 2 && steps > 2) TILE_LOAD(2, 0);
    }
    const int t1 = t0 + DMA_TABLE_TILES < steps ? t0 + DMA_TABLE_TILES : steps;
    for (int i = t0; i < t1; ++i) {
      const int K0 = my_begin + 32 * i;
      unsigned char* const tile = tile_lds + (i % TILES) * T::BYTES;
      // this wave's part of tile i has landed once only the loads of the tiles after it are left
      if (TILES > 2 && i + 2 < steps) loads_left<2 * PER>();
      else if (TILES > 2 && i + 1 < steps) loads_left<PER>();
      else loads_left<0>();
      // The bare barrier: with the fence of __syncthreads the compiler would wait here for every load it
      // knows of.  No access to memory may move across it: the next loads overwrite what other waves read
      // until here.
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (i + TILES - 1 < steps) TILE_LOAD(i + TILES - 1, t0);
      if (K0 + 31 > first_pos || K0 < open_lo) {
        const bool ok0 = pages[2 * (i - t0)] >= 0, ok1 = pages[2 * (i - t0) + 1] >= 0;
        dma_tile_products<NQK, NG, true, EXTRA, BiasPtr>(tile, K0, qreg, clo, chi, acc, m, negm, l, k_at, v_at, last_pos, ok0, ok1,
                                                         score_scale, bias_row, bias_last, EXTRA && K0 + 31 + bias_last <= first_pos);
      } else {
        dma_tile_products<NQK, NG, false, EXTRA, BiasPtr>(tile, K0, qreg, clo, chi, acc, m, negm, l, k_at, v_at, last_pos, true, true,
                                                          score_scale, bias_row, bias_last, EXTRA && K0 + 31 + bias_last <= first_pos);
      }
    }
  }
#undef TILE_LOAD
  // nothing is on its way any more, and every wave is done with the tiles: their memory serves the merge
  loads_left<0>();
  __syncthreads();
  if (KS > 1) {
    // The parts behind the first hand (reference value, sum, output) over, which the first adds in their order.  Which of a sum's two
    // products is rounded by itself is written out: left to the compiler it differs between the kernels this is part of.
    float* const w = reinterpret_cast<float*>(lds) + (size_t)wave * PER_LANE * 64 + lane;
    constexpr int PART = TEAM * PER_LANE * 64;
    if (part > 0) {
      float* const mine = w + (part - 1) * PART;
#pragma unroll
      for (int qg = 0; qg < NG; ++qg) {
#pragma unroll
        for (int n = 0; n < 2 * NQK; ++n)
#pragma unroll
          for (int e = 0; e < 4; ++e) mine[(qg * (8 * NQK + 2) + 4 * n + e) * 64] = acc[qg][n][e];
        mine[(qg * (8 * NQK + 2) + 8 * NQK) * 64] = m[qg];
        mine[(qg * (8 * NQK + 2) + 8 * NQK + 1) * 64] = l[qg];
      }
    }
    __syncthreads();
    if (part > 0) return;
#pragma unroll 1
    for (int other = 0; other < KS - 1; ++other) {
      const float* const its = w + other * PART;
#pragma unroll
      for (int qg = 0; qg < NG; ++qg) {
        const float m_b = its[(qg * (8 * NQK + 2) + 8 * NQK) * 64], l_b = its[(qg * (8 * NQK + 2) + 8 * NQK + 1) * 64];
        const float M = fmaxf(m[qg], m_b);
        const float fa = fast_exp2(m[qg] - M), fb = fast_exp2(m_b - M);
#pragma unroll
        for (int n = 0; n < 2 * NQK; ++n)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            acc[qg][n][e] = fmaf(acc[qg][n][e], fa, its[(qg * (8 * NQK + 2) + 4 * n + e) * 64] * fb);
        l[qg] = fmaf(l[qg], fa, l_b * fb);
        m[qg] = M;
      }
    }
  }
#pragma unroll
  for (int qg = 0; qg < NG; ++qg) {
    float lt = l[qg];
    lt = sum_with_lane_xor32(sum_with_lane_xor16(lt));
    if (chi[qg] < 0) continue;
    if constexpr (EXTRA) lt += sink_of(extras, head, m[qg]);
    float inv = lt > 0.f ? 1.f / lt : 0.f;
    if constexpr (EXTRA) inv *= gate_of(extras, tok[qg], head);
    bf16_t* op = out + (size_t)tok[qg] * out_stride + (size_t)head * HD;
#pragma unroll
    for (int n = 0; n < 2 * NQK; ++n)
      *reinterpret_cast<uint2*>(op + 16 * n + 4 * g) =
          make_uint2(pack2_bf16(acc[qg][n][0] * inv, acc[qg][n][1] * inv),
                     pack2_bf16(acc[qg][n][2] * inv, acc[qg][n][3] * inv));
  }
