// Attention in 32 bits on the matrix cores (v_mfma_f32_16x16x4_f32), for heads whose keys and values come in steps of 16
// channels: part of attention.hip, which has the sizes, the arguments and what they mean (AttnArgs).
//
// A wave takes tiles of 16 keys and C tiles of 16 columns, a column being a query row and one head of the key/value
// head's group.  Scores come transposed, S^T[key][column] = K . Q^T: lane l holds key l % 16 of the first operand at
// channels 16 c + 4 (l / 16) + j, instruction j, 16 bytes a load, and S^T[4 (l / 16) + e][l % 16] of the result.  That is
// what the second product wants of its second operand, O^T = V^T . P^T, if its instruction e takes the keys 4 g + e of
// the lane groups g: nothing is moved between lanes, and a lane's 16 bytes of a value channel are those keys.
//
// Measured, microseconds, against a wave a (token, head) (attention_rows_kernel): 8 single tokens of 100 to 905 keys on 9/3
// heads of 64 10.4 (31), 8 of 2,000 keys on 32/32 heads 42 (84; 48 at 5.5 TB/s if nothing came from a cache); a prompt of
// 509 tokens on 32/4 heads of 64 28 (155), of 2,000 on 32/8 heads of 128 450 (4,990; 73 TFLOP/s counted causally; 27 and 416
// without the search for values that are no numbers).  Over a prompt the products bound it (a tile of keys is 32
// instructions of 32 cycles a column tile at 64 channels, beside 130 vector instructions); over single tokens the trips to
// memory.  Measured and no faster: 8 waves a block (28 and 204 against 26 and 200 at 509 and 2,000 tokens), three and four
// tiles in registers, a tile's scores taken ahead of the softmax of the tile before it (31 and 255), such values added behind
// the products from memory again (31 fewer registers; 28 and 453 where this takes 28 and 450).
#pragma once

typedef __attribute__((ext_vector_type(4))) float attn_f32x4;

constexpr int kF32Waves = 4;                     // of a block: they deal the item's tiles of keys and merge in LDS
constexpr int kF32Columns = HDR <= 128 ? 2 : 1;  // column tiles of an item of a prompt (registers)
constexpr bool kF32Ahead = HDR <= 64;            // the next tile's keys and values asked for under this one's products
constexpr float kF32Rise = 8.0f;                 // the softmax reference moves when a score rises this far above it

struct F32Step {
  // a prompt's items: tile_seq / tile_row0 name a sequence of the step and the first of an item's rows; null for a
  // step of single tokens, whose items are the tokens
  const int* tile_seq;
  const int* tile_row0;
  const int* seq_slot;
  const int* seq_start;
  const int* seq_pos0;
  int chunks;      // items a key/value head's group is cut into
  int splits;      // blocks an item's keys are cut into (single tokens only)
  float* partial;  // [tokens][heads][splits][kF32Partial], with splits > 1
};
constexpr int kF32Partial = HDV + 4;

// (two waves a SIMD up to 64 channels: left to itself the compiler takes 260 registers)
template <int C, bool SINGLE>
__global__ __launch_bounds__(kWave * kF32Waves, kF32Ahead ? 2 : 1) void attention_f32_kernel(AttnArgs a, F32Step step) {
  constexpr int KC = HD / 16, VC = HDV / 16;
  constexpr int kOutRow = 64 + 4;  // floats of a column's 64 channels in LDS
  __shared__ float merged[kF32Waves][16][kOutRow];
  __shared__ float state[kF32Waves][C * 16][2];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int r = lane % 16, g = lane / 16;
  const int group = a.heads / a.kv_heads;
  const int per_item = a.kv_heads * step.chunks;
  const int item = blockIdx.x / per_item, kv_head = blockIdx.x % per_item / step.chunks, chunk = blockIdx.x % step.chunks;

  // The item's columns.  A row beyond the sequence's last computes what the last one does, and is not stored; so
  // is a head beyond the group's.
  int slot, first_token, rows, first_pos;  // the item's rows are tokens first_token .. + rows - 1 at positions first_pos ..
  if constexpr (SINGLE) {
    slot = a.tok_slot[item];
    first_token = item;
    rows = 1;
    first_pos = slot < 0 ? 0 : a.tok_pos[item];
  } else {
    const int seq = step.tile_seq[item], row0 = step.tile_row0[item];
    const int start = step.seq_start[seq], count = step.seq_start[seq + 1] - start;
    if (row0 >= count) return;  // (an item that fills a list up)
    slot = step.seq_slot[seq];
    first_token = start + row0;
    const int most = group == 1 ? 16 * C : 16;
    rows = count - row0 < most ? count - row0 : most;
    first_pos = step.seq_pos0[seq] + row0;
  }
  auto column_row = [&](int t, int q) { return SINGLE ? 0 : (group == 1 ? t * 16 + q : q); };
  auto column_head = [&](int t, int q) {  // within the group
    return SINGLE ? (chunk * C + t) * 16 + q : (group == 1 ? 0 : chunk * C + t);
  };
  if (slot < 0) {  // padding rows of a step that runs from fixed buffers
    if (SINGLE && step.splits == 1)
      for (int at = threadIdx.x; at < C * 16 * HDV; at += blockDim.x) {
        const int head = column_head(at / HDV / 16, at / HDV % 16);
        if (head < group) ((float*)a.out)[((size_t)item * a.heads + kv_head * group + head) * HDV + at % HDV] = 0.0f;
      }
    return;
  }

  attn_f32x4 q[C][KC];
  int pos[C], lo[C], head[C];
#pragma unroll
  for (int t = 0; t < C; ++t) {
    int row = column_row(t, r), h = column_head(t, r);
    row = row < rows ? row : rows - 1;
    h = h < group ? h : group - 1;
    pos[t] = first_pos + row;
    lo[t] = first_seen(a.window, pos[t]);
    head[t] = kv_head * group + h;
    const float* from = (const float*)a.q + ((size_t)(first_token + row) * a.heads + head[t]) * HD + g * 4;
#pragma unroll
    for (int c = 0; c < KC; ++c) q[t][c] = *(const attn_f32x4*)(from + c * 16);
  }

  // Tiles of 16 keys, in this order: the kept first ones that the window has left behind, those that a row sees,
  // pooled blocks.  The waves of the item's blocks take them in turn.
  const int last_pos = first_pos + rows - 1;
  const int lo_first = first_seen(a.window, first_pos), lo_last = first_seen(a.window, last_pos);
  const int near0 = lo_first / 16, near1 = last_pos / 16 + 1;
  const int kept = min((a.keep_first + 15) / 16, near0);
  const int pooled = a.pool > 0 ? (lo_last / a.pool + 15) / 16 : 0;
  const int tiles = kept + near1 - near0 + pooled;
  const int stride = SINGLE ? kF32Waves * step.splits : kF32Waves;
  auto tile_of = [&](int i) { return i < kept ? i : (i < tiles - pooled ? near0 + i - kept : i - (tiles - pooled)); };
  auto page_of = [&](int i) {
    const int* table = i < tiles - pooled ? a.block_table + (size_t)slot * a.max_pages : a.pool_table + (size_t)slot * a.pool_max_pages;
    return table[tile_of(i) / 4];
  };
  struct Operands {
    attn_f32x4 k[KC], v[VC];
  };
  auto load = [&](Operands& into, int i, int page) {
    const bool near = i < tiles - pooled;
    const int in_page = tile_of(i) % 4 * 16;  // the tile's first token of its page
    const float* keys = (const float*)(near ? a.k_pages : a.pool_k) + ((size_t)page * a.kv_heads + kv_head) * nnis_k_page_elems(HD);
    const float* values = (const float*)(near ? a.v_pages : a.pool_v) + ((size_t)page * a.kv_heads + kv_head) * nnis_v_page_elems(HDV);
    keys += nnis_k_offset(in_page + r, g * 4);
    values += nnis_v_offset(r, in_page + g * 4);
#pragma unroll
    for (int c = 0; c < KC; ++c) into.k[c] = *(const attn_f32x4*)(keys + nnis_k_offset(0, c * 16));
#pragma unroll
    for (int c = 0; c < VC; ++c) into.v[c] = *(const attn_f32x4*)(values + nnis_v_offset(c * 16, 0));
  };

  float ref[C], sum[C];
  attn_f32x4 out[C][VC];
#pragma unroll
  for (int t = 0; t < C; ++t) {
    ref[t] = -INFINITY;
    sum[t] = 0.0f;
#pragma unroll
    for (int c = 0; c < VC; ++c) out[t][c] = (attn_f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  }
  auto take = [&](Operands& kv, int i) {
    // Two chains of products a score, so that none waits for the one before it, over 64 channels at a time: a chain rounds
    // after each of its products.  (Relative error against 64 bits at 64 / 128 / 256 channels over 2,000 keys: 5.0e-7 / 4.8e-7 /
    // 4.5e-7 over a prompt and 6.5e-7 / 6.3e-7 / 5.8e-7 for single tokens in one block; the row kernel 7.4e-7 / 9.9e-7 / 1.4e-6.)
    attn_f32x4 s[C], even[C], odd[C];
#pragma unroll
    for (int c = 0; c < KC; ++c) {
#pragma unroll
      for (int t = 0; t < C; ++t)
        if (c % 4 == 0) even[t] = odd[t] = (attn_f32x4){0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < 4; j += 2)
#pragma unroll
        for (int t = 0; t < C; ++t) {
          even[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv.k[c][j], q[t][c][j], even[t], 0, 0, 0);
          odd[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv.k[c][j + 1], q[t][c][j + 1], odd[t], 0, 0, 0);
        }
#pragma unroll
      for (int t = 0; t < C; ++t)
        if (c % 4 == 3 || c == KC - 1) s[t] = c < 4 ? even[t] + odd[t] : s[t] + (even[t] + odd[t]);
    }
    const bool near = i < tiles - pooled;
    const int key0 = tile_of(i) * 16;
    const bool masked = !near || key0 + 15 > first_pos || key0 < lo_last;  // else every row sees every key of the tile
    const int valid = near ? last_pos + 1 : lo_last / a.pool;  // keys from here on are not the sequence's: what lies there may be no number
    if (key0 + 16 > valid) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool held = key0 + 4 * g + e < valid;
#pragma unroll
        for (int c = 0; c < VC; ++c) kv.v[c][e] = held ? kv.v[c][e] : 0.0f;
      }
    }
    auto seen = [&](int t, int key) { return near ? key <= pos[t] && (key >= lo[t] || key < a.keep_first) : key < lo[t] / a.pool; };
    bool rises = false;
#pragma unroll
    for (int t = 0; t < C; ++t) {
      s[t] *= a.scale;
      if (a.softcap > 0.0f) {
#pragma unroll
        for (int e = 0; e < 4; ++e) s[t][e] = a.softcap * tanhf(s[t][e] / a.softcap);
      }
      if (a.bias && near) {
#pragma unroll
        for (int e = 0; e < 4; ++e) s[t][e] += a.bias[(size_t)head[t] * (a.reach + 1) + max(0, min(pos[t] - (key0 + 4 * g + e), a.reach))];
      }
      if (a.terms.r1 && near) {
#pragma unroll
        for (int e = 0; e < 4; ++e) s[t][e] -= a.terms.r1[head[t]] * log1pf(a.terms.r2[head[t]] * (float)max(0, pos[t] - (key0 + 4 * g + e)));
      }
      if (masked) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s[t][e] = seen(t, key0 + 4 * g + e) ? s[t][e] : -INFINITY;
        }
      }
      rises |= fmaxf(fmaxf(s[t][0], s[t][1]), fmaxf(s[t][2], s[t][3])) > ref[t] + kF32Rise;
    }
    if (__any(rises)) {
#pragma unroll
      for (int t = 0; t < C; ++t) {
        float m = fmaxf(fmaxf(s[t][0], s[t][1]), fmaxf(s[t][2], s[t][3]));
        m = fmaxf(m, __shfl_xor(m, 16, kWave));
        m = fmaxf(fmaxf(m, __shfl_xor(m, 32, kWave)), ref[t]);
        const float factor = ref[t] == -INFINITY ? 0.0f : expf(ref[t] - m);  // (nothing is held yet)
        ref[t] = m;
        sum[t] *= factor;
#pragma unroll
        for (int c = 0; c < VC; ++c) out[t][c] *= factor;
      }
    }
#pragma unroll
    for (int t = 0; t < C; ++t) {
      const float against = ref[t] == -INFINITY ? 0.0f : ref[t];  // (a column that has seen no key yet: its weights are zeros)
#pragma unroll
      for (int e = 0; e < 4; ++e) s[t][e] = expf(s[t][e] - against);
      sum[t] += (s[t][0] + s[t][1]) + (s[t][2] + s[t][3]);
    }
    // A value that is infinite or no number, times the weight of a row that does not see its key, zero, would be no number: of a
    // tile that some rows see a part of, such values are added to the rows that see them here, and count as zeros below.
    if (masked) {
      attn_f32x4 none = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int c = 0; c < VC; ++c) none += kv.v[c] * 0.0f;
      if (__builtin_expect(__any(!((none[0] + none[1]) + (none[2] + none[3]) == 0.0f)), 0)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll 1
          for (int k4 = 0; k4 < 4; ++k4)  // the key 4 k4 + e: its weights lie in the lane group k4, as its values do
#pragma unroll
            for (int t = 0; t < C; ++t) {
              const float weight = __shfl(s[t][e], k4 * 16 + r, kWave);
              const bool counts = seen(t, key0 + 4 * k4 + e);
#pragma unroll
              for (int c = 0; c < VC; ++c) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                  const float value = __shfl(kv.v[c][e], k4 * 16 + 4 * g + i, kWave);
                  out[t][c][i] = counts && !(value * 0.0f == 0.0f) ? fmaf(weight, value, out[t][c][i]) : out[t][c][i];
                }
                __builtin_amdgcn_sched_barrier(0);  // (one channel tile after another: registers)
              }
            }
#pragma unroll
          for (int c = 0; c < VC; ++c) kv.v[c][e] = kv.v[c][e] * 0.0f == 0.0f ? kv.v[c][e] : 0.0f;
        }
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int c = 0; c < VC; ++c)
#pragma unroll
        for (int t = 0; t < C; ++t) out[t][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv.v[c][e], s[t][e], out[t][c], 0, 0, 0);
  };

  int i = (SINGLE ? blockIdx.y * kF32Waves : 0) + wave;
  if (i < tiles) {
    int page = page_of(i);
    if constexpr (kF32Ahead) {
      // two sets of operands in turn: a tile's are asked for before the one before it is multiplied, its page's number a
      // tile earlier (beyond the last tile the one at hand again: valid memory, never used)
      Operands one, other;
      auto held = [&](int at) { return at < tiles ? at : i; };
      load(one, i, page);
      int next = held(i + stride);
      page = page_of(next);
      while (true) {
        load(other, next, page);
        const int behind = held(i + 2 * stride);
        page = page_of(behind);
        take(one, i);
        i += stride;
        if (i >= tiles) break;
        load(one, behind, page);
        next = held(i + 2 * stride);
        page = page_of(next);
        take(other, i);
        i += stride;
        if (i >= tiles) break;
      }
    } else {
      Operands one;
      for (; i < tiles; i += stride) {
        load(one, i, page);
        page = page_of(i + stride < tiles ? i + stride : i);
        take(one, i);
      }
    }
  }

  // The waves meet: references and sums first, then the outputs, 64 channels of a column tile at a time.
#pragma unroll
  for (int t = 0; t < C; ++t) {
    sum[t] += __shfl_xor(sum[t], 16, kWave);
    sum[t] += __shfl_xor(sum[t], 32, kWave);
    if (g == 0) {
      state[wave][t * 16 + r][0] = ref[t];
      state[wave][t * 16 + r][1] = sum[t];
    }
  }
  __syncthreads();
  const bool whole = !SINGLE || step.splits == 1;
#pragma unroll
  for (int t = 0; t < C; ++t) {
    auto reference = [&](int column, int of_head) {
      float m = whole && a.sink ? a.sink[of_head] : -INFINITY;
#pragma unroll
      for (int w = 0; w < kF32Waves; ++w) m = fmaxf(m, state[w][column][0]);
      return m;
    };
    const float m_lane = reference(t * 16 + r, head[t]);
    const float weight = ref[t] == -INFINITY ? 0.0f : expf(ref[t] - m_lane);
    // the thread's four channels of a column in each round
    const int at_q = threadIdx.x / 16, at_c = threadIdx.x % 16 * 4;
    const int row = column_row(t, at_q), h = column_head(t, at_q);
    const bool stored = row < rows && h < group;
    const int of_head = kv_head * group + (h < group ? h : group - 1);
    const size_t token = first_token + (row < rows ? row : rows - 1);
    const float m = reference(t * 16 + at_q, of_head);
    float total = whole && a.sink ? expf(a.sink[of_head] - m) : 0.0f;
#pragma unroll
    for (int w = 0; w < kF32Waves; ++w) {
      const float m_w = state[w][t * 16 + at_q][0];
      total += m_w == -INFINITY ? 0.0f : state[w][t * 16 + at_q][1] * expf(m_w - m);
    }
    const float factor = whole ? (a.terms.gate ? head_gate(a.terms, token, of_head) : 1.0f) / total : 1.0f;
    float* to = whole ? (float*)a.out + (token * a.heads + of_head) * HDV
                      : step.partial + ((token * a.heads + of_head) * step.splits + blockIdx.y) * kF32Partial;
#pragma unroll
    for (int c0 = 0; c0 < VC; c0 += 4) {
      if (t + c0 > 0) __syncthreads();  // what the round before left there has been read
#pragma unroll
      for (int c = c0; c < (c0 + 4 < VC ? c0 + 4 : VC); ++c) *(attn_f32x4*)&merged[wave][r][(c - c0) * 16 + g * 4] = out[t][c] * weight;
      __syncthreads();
      if (stored && c0 * 16 + at_c < HDV) {
        attn_f32x4 v = *(const attn_f32x4*)&merged[0][at_q][at_c];
#pragma unroll
        for (int w = 1; w < kF32Waves; ++w) v += *(const attn_f32x4*)&merged[w][at_q][at_c];
        *(attn_f32x4*)(to + c0 * 16 + at_c) = v * factor;
      }
    }
    if (!whole && stored && at_c == 0) {
      to[HDV] = m;
      to[HDV + 1] = total;
    }
  }
}

// The blocks of one (token, head): out = sum_s O_s e^(m_s - M) / (sum_s l_s e^(m_s - M) + e^(sink - M)).
__global__ void attention_f32_combine_kernel(AttnArgs a, F32Step step) {
  const int token = blockIdx.x, head = blockIdx.y;
  float* out = (float*)a.out + ((size_t)token * a.heads + head) * HDV;
  if (a.tok_slot[token] < 0) {
    for (int d = threadIdx.x; d < HDV; d += blockDim.x) out[d] = 0.0f;
    return;
  }
  const float* base = step.partial + ((size_t)token * a.heads + head) * step.splits * kF32Partial;
  constexpr int kMost = 16;
  float m[kMost], l[kMost];
  const float sink = a.sink ? a.sink[head] : -INFINITY;
  float m_all = sink;
#pragma unroll
  for (int s = 0; s < kMost; ++s) {  // (beyond the last: the last again, not counted)
    const float* p = base + (size_t)(s < step.splits ? s : step.splits - 1) * kF32Partial;
    m[s] = p[HDV];
    l[s] = p[HDV + 1];
    m_all = fmaxf(m_all, m[s]);
  }
  float total = a.sink ? expf(sink - m_all) : 0.0f;
#pragma unroll
  for (int s = 0; s < kMost; ++s) {
    m[s] = s >= step.splits || m[s] == -INFINITY ? 0.0f : expf(m[s] - m_all);
    total += l[s] * m[s];
  }
  const float factor = (a.terms.gate ? head_gate(a.terms, token, head) : 1.0f) / total;
  for (int d = threadIdx.x; d < HDV; d += blockDim.x) {
    float v = 0.0f;
#pragma unroll
    for (int s = 0; s < kMost; ++s) v += base[(size_t)(s < step.splits ? s : step.splits - 1) * kF32Partial + d] * m[s];
    out[d] = v * factor;
  }
}
constexpr int kF32MostSplits = 16;
