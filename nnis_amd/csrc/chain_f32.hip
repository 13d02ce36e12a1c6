// The layers of a step of few single tokens in one launch, in 32 bits: chain.hip's stages on v_mfma_f32_16x16x4_f32, for weights
// in the checkpoint's order (as gemm_f32.hip's kernel for few rows takes them: 16 bytes a lane are 16 k of 16 rows).
//
// Rows are exchanged by strips of 16 channels, [strip][row][16], 64 bytes that one block writes.  A strip of the stream's rows, which is
// times the next norm's gain, has the rows' parts of their sums of squares behind it (a word a row, 4, 8 or 16 of them); the stream
// itself, [strip][row][16], lies apart.  The row's scale comes behind the product.
//
// A block is a unit of a product (a pair of strips of 16 weight rows, or a strip) and has 8 waves, wave w the chunks of 16 k w, w + 8, ..;
// WIDE (from a width of 1,025 on): more registers of weights a wave, one block a compute unit.  Bound by the way from a stage's
// stores to the next one's loads (1 to 2 us, five stages a layer) and, wide, by the weights' way in.  Whole steps in microseconds, by
// the layers' kernels and by this launch: 30 layers of width 576, 9/3 heads, batch 1 behind 60 / 370 / 1,000 tokens 879 / 1,008 / 1,018
// and 530 / 586 / 590, batch 8 1,071 / 1,090 / 1,134 and 572 / 624 / 660, batch 16 1,296 / 1,344 / 1,425 and 634 / 705 / 761; 22
// layers of width 2,048, 32/4 heads (4.4 GB of weights: 0.9 ms of copy), batch 1 and 8 behind 300: 1,433 and 1,566 and 1,286 and 1,426.
#include <hip/hip_runtime.h>

#include "chain.h"

namespace {

constexpr int HD = kChainHead, kWaves = 8;
constexpr int kRow32 = 16;  // words of a row's strip
constexpr float kRise = 8.0f;  // as in attention_f32.h: the softmax reference moves when a score rises this far above it

struct ChainLayer32 {
  const float *w_qkv, *w_o, *w_gate_up, *w_down;
  const float *gain1, *gain2;
  float *k_pages, *v_pages;
};

struct ChainArgs32 {
  const ChainLayer32* layers;
  int layer_count, m, width, heads, kv_heads, inner, splits;
  float eps, scale, inv_width;
  const float* x;  // [m, width]
  float *x_out, *y_out;  // [m, width]: the stream behind the last attention, and what the last feed-forward adds to it
  const float *tok_cos, *tok_sin;
  const int *tok_pos, *tok_page, *tok_pages;
  int max_pages;
  unsigned *words, *run_words;
  unsigned words_bytes, run_bytes, layer_words, layer_runs;
  unsigned stream1, stream2, plain1, plain2, q, k, v, attn, act;  // where a layer's words lie
  unsigned strip_words;  // of the stream's rows as the next product takes them
  int n_strip, n_entry, n_qkv, n_att, n_comb, n_gate;  // blocks of a stage (the output projection and down: a strip each)
  unsigned *fail, *host_fail;
};

__device__ __forceinline__ u32x4 marked4(f32x4 v) { return (u32x4){marked(v[0]), marked(v[1]), marked(v[2]), marked(v[3])}; }

template <int ROWS>
struct Shared32 {
  union {
    struct {
      f32x4 acc[kWaves][2][kWave];
      float squares[kWaves][kMostRows];  // WIDE
      RowScales<ROWS> scales;            // not WIDE
    } product;
    struct {
      __attribute__((aligned(16))) float o[kWaves][16][HD + 4];  // a head's outputs, then its sum
      float m[kWaves][16], weights[kWaves][16][kWaves];
    } attention;
  };
};

// STRIPS strips of 16 weight rows times the step's rows.  A wave asks for the weights of its first STEPS chunks when the block
// begins; XB chunks of the operand are asked for together.  A step of the operand beyond the last chunk reads the last again
// and is not multiplied.
// NORM: a row that a norm prepared, whose parts of the sum of squares each wave takes with its own chunks (SUMS), or all of them, with
// its first trip, for the last wave.
template <int ROWS, int STRIPS, int STEPS, int XB, bool NORM, bool SUMS>
struct Product32 {
  static_assert(STEPS % XB == 0, "whole trips");
  f32x4 w[STEPS][STRIPS], acc[STRIPS][4];  // a sum for each of a lane's four k: shorter chains (K 8,256: 0.69 to 0.88 of the layers' error
                                             // against 64 bits over whole models of two layers; one sum for all 1.17 to 1.29)
  const float* row[STRIPS];
  float square;
  int chunks, wave, lane;

  __device__ __forceinline__ void ask(int base) {
#pragma unroll
    for (int d = 0; d < STEPS; ++d) {
      if (base + d * kWaves >= chunks) continue;  // (the same for the whole wave)
#pragma unroll
      for (int j = 0; j < STRIPS; ++j) w[d][j] = __builtin_nontemporal_load((const f32x4*)(row[j] + (base + d * kWaves) * 16));
    }
  }
  // first_row(j): the first weight row of strip j
  template <typename Row>
  __device__ __forceinline__ void begin(const float* weight, Row first_row, int k, int lane_, int wave_) {
    lane = lane_;
    wave = wave_;
    square = 0.0f;
    chunks = k / 16;
#pragma unroll
    for (int j = 0; j < STRIPS; ++j) {
      row[j] = weight + (size_t)(first_row(j) + lane % 16) * k + lane / 16 * 4;
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[j][e] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    }
    ask(wave);
  }
  // the operand: the lane's row begins at byte `row_at`, `stride` bytes from strip to strip; `sums`: the first strip's sums' first word
  __device__ __forceinline__ void run(const Exchange& ex, Shared32<ROWS>& s, unsigned row_at, unsigned stride, unsigned sums, int row, float inv_width, float eps) {
    const unsigned at = row_at + lane / 16 * 16, sum_at = (sums + row) * 4;
    constexpr int kMore = NORM && !SUMS ? RowScales<ROWS>::kFours : 0;
    u32x4 more[kMore > 0 ? kMore : 1];
    auto ask_more = [&](int i) { return RowScales<ROWS>::at(i, lane, sums, stride, chunks); };
    for (int base = wave; base < chunks; base += kWaves * STEPS) {
      if (base != wave) ask(base);
#pragma unroll
      for (int b = 0; b < STEPS; b += XB) {
        if (base + b * kWaves >= chunks) continue;
        u32x4 v[XB + kMore];
        unsigned part[XB];
        auto chunk = [&](int d) { return (unsigned)min(base + (b + d) * kWaves, chunks - 1) * stride; };
        auto pieces = [&](int d) { return d < XB ? At{at, chunk(d)} : ask_more(d - XB); };
        if constexpr (NORM && SUMS) ex.take(v, pieces, part, [&](int d) { return At{sum_at, chunk(d)}; });
        else ex.take(v, pieces);
        if constexpr (kMore > 0) {
#pragma unroll
          for (int i = 0; i < kMore; ++i) more[i] = v[XB + i];
        }
#pragma unroll
        for (int d = 0; d < XB; ++d) {
          if (base + (b + d) * kWaves >= chunks) continue;
          const f32x4 x = __builtin_bit_cast(f32x4, v[d]);
          if constexpr (NORM && SUMS) square += __uint_as_float(part[d]);
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int j = 0; j < STRIPS; ++j) acc[j][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[b + d][j][e], x[e], acc[j][e], 0, 0, 0);
        }
      }
    }
    if constexpr (kMore > 0) {
      if (wave == kWaves - 1) {
        if (wave >= chunks) ex.take(more, ask_more);  // (it had no product)
        s.product.scales.make(more, lane, chunks, inv_width, eps);
      }
    }
  }
  // the waves' sums added up in their order; false for the waves that are done.  scale: of the lane's row (NORM)
  __device__ __forceinline__ bool finish(Shared32<ROWS>& s, const Ends<ROWS>& ends, Floats<Ends<ROWS>::kEach> (&sums)[STRIPS], float& scale, float eps) {
    constexpr int kEach = Ends<ROWS>::kEach;
#pragma unroll
    for (int j = 0; j < STRIPS; ++j) s.product.acc[wave][j][lane] = (acc[j][0] + acc[j][1]) + (acc[j][2] + acc[j][3]);
    if constexpr (NORM && SUMS) {
      if (lane < 16) s.product.squares[wave][lane] = square;
    }
    __syncthreads();
    if (wave != 0) return false;
#pragma unroll
    for (int j = 0; j < STRIPS; ++j) {
      auto part_at = [&](int p) { return load_floats<kEach>((const float*)&s.product.acc[p][j][ends.from] + ends.first % 4); };
      sums[j] = part_at(0);
#pragma unroll
      for (int p = 1; p < kWaves; ++p) {
        const Floats<kEach> part = part_at(p);
#pragma unroll
        for (int e = 0; e < kEach; ++e) sums[j][e] += part[e];
      }
    }
    if constexpr (NORM && SUMS) {
      float total = s.product.squares[0][ends.row];
#pragma unroll
      for (int p = 1; p < kWaves; ++p) total += s.product.squares[p][ends.row];
      scale = 1.0f / sqrtf(total / (float)(chunks * 16) + eps);
    } else if constexpr (NORM) {
      scale = s.product.scales.scale[ends.row];
    }
    return true;
  }
};

// a word of some row of the stream's strips at `first_word`
__device__ __forceinline__ unsigned a_row(const ChainArgs32& a, unsigned first_word, int some) {
  return first_word + some / a.m % a.n_strip * a.strip_words + some % a.m * kRow32;
}

template <int ROWS>
__device__ __forceinline__ void entry_stage(const ChainArgs32& a, const Exchange& ex, int row) {
  for (int c = threadIdx.x * 4; c < a.width; c += kWave * kWaves * 4) {  // (a strip's four lanes come together: the width is whole strips)
    const f32x4 v = *(const f32x4*)(a.x + (size_t)row * a.width + c), gain = *(const f32x4*)(a.layers[0].gain1 + c);
    float part = (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]);
    part += __shfl_xor(part, 1, kWave);
    part += __shfl_xor(part, 2, kWave);
    const int strip = c / 16, four = c % 16 / 4;
    const unsigned word = a.stream1 + strip * a.strip_words;
    ex.put(word + row * kRow32 + 4 * four, marked4(v * gain));
    ex.put(a.plain1 + (strip * a.m + row) * kRow32 + 4 * four, marked4(v));
    if (four == 0)  // the last row's also in place of rows that there are none of
      for (int to = row; to < (row + 1 < a.m ? row + 1 : sum_words(ROWS)); ++to) ex.put(word + a.m * kRow32 + to, marked(part));
  }
}

template <bool WIDE, int ROWS>
__device__ __forceinline__ void qkv_stage(const ChainArgs32& a, const Exchange& ex, Shared32<ROWS>& s, int layer, int unit) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, r = lane % 16;
  const ChainLayer32& L = a.layers[layer];
  const unsigned here = layer * a.layer_words;
  const int head = unit / 2, f0 = unit % 2 * 16;  // channels f0 .. f0 + 15 of the head and those half a head on
  constexpr int kSteps = WIDE ? 16 : 6, kTogether = WIDE ? 8 : 6;
  constexpr int kEach = Ends<ROWS>::kEach;
  Product32<ROWS, 2, kSteps, kTogether, true, WIDE> p;
  p.begin(L.w_qkv, [&](int j) { return head * HD + f0 + j * (HD / 2); }, a.width, lane, wave);
  const Ends<ROWS> ends(lane);
  const int row = min(ends.row, a.m - 1), f = f0 + ends.first, operand_row = min(r, a.m - 1);
  const Floats<kEach> c = load_floats<kEach>(a.tok_cos + row * (HD / 2) + f), sn = load_floats<kEach>(a.tok_sin + row * (HD / 2) + f);
  const int pos = a.tok_pos[row], page = a.tok_page[row];
  ex.template gate<true>(a_row(a, here + a.stream1, unit * 61), wave);
  p.run(ex, s, (here + a.stream1 + operand_row * kRow32) * 4, a.strip_words * 4, here + a.stream1 + a.m * kRow32, operand_row, a.inv_width, a.eps);
  Floats<kEach> sums[2], out_lo, out_hi;
  float scale;
  if (!p.finish(s, ends, sums, scale, a.eps)) return;
  if (ends.row >= a.m) return;
#pragma unroll
  for (int e = 0; e < kEach; ++e) {
    const float lo = sums[0][e] * scale, hi = sums[1][e] * scale;
    out_lo[e] = lo;
    out_hi[e] = hi;
    if (head < a.heads + a.kv_heads) {
      out_lo[e] = lo * c[e] - hi * sn[e];
      out_hi[e] = hi * c[e] + lo * sn[e];
    }
  }
  unsigned to;  // [head][strip][row]
  if (head < a.heads) to = a.q + head * a.m * HD;
  else if (head < a.heads + a.kv_heads) to = a.k + (head - a.heads) * a.m * HD;
  else to = a.v + (head - a.heads - a.kv_heads) * a.m * HD;
  to += here + (f0 / 16 * a.m + row) * 16 + ends.first;
  put_floats(ex, to, out_lo);
  put_floats(ex, to + HD / 32 * a.m * 16, out_hi);
  if (page < 0 || head < a.heads) return;
  const int in_page = pos % kPageTokens;
  if (head < a.heads + a.kv_heads) {
    float* dst = L.k_pages + ((size_t)page * a.kv_heads + head - a.heads) * nnis_k_page_elems(HD);
#pragma unroll
    for (int e = 0; e < kEach; ++e) {  // (a lane's channels lie within a chunk of 8)
      dst[nnis_k_offset(in_page, f) + e] = out_lo[e];
      dst[nnis_k_offset(in_page, f + HD / 2) + e] = out_hi[e];
    }
  } else {
    float* dst = L.v_pages + ((size_t)page * a.kv_heads + head - a.heads - a.kv_heads) * nnis_v_page_elems(HD);
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
      dst[nnis_v_offset(f + e, in_page)] = out_lo[e];
      dst[nnis_v_offset(f + HD / 2 + e, in_page)] = out_hi[e];
    }
  }
}

// A run of a sequence's keys against the query heads of a key head (up to 16: the columns), in tiles of 16 keys (attention_f32.h:
// the same products in the same layouts).  The pages hold every key but the step's own, which comes from the exchange and takes
// its place in its tile's operands.
template <int ROWS>
__device__ __forceinline__ void attention_stage(const ChainArgs32& a, const Exchange& ex, Shared32<ROWS>& s, int layer, int item) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, r = lane % 16, g = lane / 16;
  const ChainLayer32& L = a.layers[layer];
  const unsigned here = layer * a.layer_words;
  const int group = a.heads / a.kv_heads;
  const int kv_head = item % a.kv_heads, token = item / a.kv_heads % a.m, split = item / (a.kv_heads * a.m);
  const int pos = a.tok_page[token] < 0 ? 0 : a.tok_pos[token];  // a padding row reads its own key only
  const int* pages = a.tok_pages + (size_t)token * a.max_pages;
  const int tiles = pos / 16 + 1, stride = kWaves * a.splits;
  const float* k_base = L.k_pages + (size_t)kv_head * nnis_k_page_elems(HD);
  const float* v_base = L.v_pages + (size_t)kv_head * nnis_v_page_elems(HD);
  const size_t k_stride = (size_t)a.kv_heads * nnis_k_page_elems(HD), v_stride = (size_t)a.kv_heads * nnis_v_page_elems(HD);
  struct Tile {
    f32x4 k[HD / 16], v[HD / 16];
  };
  auto load_keys = [&](Tile& t, int tile) {
    const float* from = k_base + (size_t)__builtin_amdgcn_readfirstlane(pages[tile / 4]) * k_stride + nnis_k_offset(tile % 4 * 16 + r, g * 4);
#pragma unroll
    for (int c = 0; c < HD / 16; ++c) t.k[c] = *(const f32x4*)(from + nnis_k_offset(0, c * 16));
  };
  auto load_values = [&](Tile& t, int tile) {
    const float* from = v_base + (size_t)__builtin_amdgcn_readfirstlane(pages[tile / 4]) * v_stride + nnis_v_offset(r, tile % 4 * 16 + g * 4);
#pragma unroll
    for (int c = 0; c < HD / 16; ++c) t.v[c] = *(const f32x4*)(from + nnis_v_offset(c * 16, 0));
  };
  // two tiles of a wave are in registers before the queries exist
  int i = split * kWaves + wave;
  Tile one, other;
  if (i < tiles) {
    load_keys(one, i);
    load_values(one, i);
  }
  if (i + stride < tiles) {
    load_keys(other, i + stride);
    load_values(other, i + stride);
  }
  ex.template gate<true>(a_row(a, here + a.stream1, item * 61), wave);
  const int head = kv_head * group + (r < group ? r : 0);
  f32x4 q[HD / 16], own_k[HD / 16];
  float own_v[HD / 16];
  {
    const unsigned strips = a.m * 64;
    const unsigned q_at = (here + a.q + (head * (HD / 16) * a.m + token) * 16 + 4 * g) * 4, k_at = (here + a.k + (kv_head * (HD / 16) * a.m + token) * 16 + 4 * g) * 4,
                   v_at = (here + a.v + (kv_head * (HD / 16) * a.m + token) * 16 + r) * 4;
    if (pos / 16 % stride == i) {  // this wave has the step's own key
      u32x4 got[2 * HD / 16];
      unsigned got_v[HD / 16];
      ex.take(got, [&](int c) { return c < HD / 16 ? At{q_at, c * strips} : At{k_at, (c - HD / 16) * strips}; }, got_v, [&](int c) { return At{v_at, c * strips}; });
#pragma unroll
      for (int c = 0; c < HD / 16; ++c) {
        q[c] = __builtin_bit_cast(f32x4, got[c]);
        own_k[c] = __builtin_bit_cast(f32x4, got[HD / 16 + c]);
        own_v[c] = __uint_as_float(got_v[c]);
      }
    } else if (i < tiles) {
      u32x4 got[HD / 16];
      ex.take(got, [&](int c) { return At{q_at, c * strips}; });
#pragma unroll
      for (int c = 0; c < HD / 16; ++c) q[c] = __builtin_bit_cast(f32x4, got[c]);
    }
  }
  f32x4 o[HD / 16];
#pragma unroll
  for (int c = 0; c < HD / 16; ++c) o[c] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  float reference = -INFINITY, sum = 0.0f;
  auto take_tile = [&](Tile& t) {
    const int key0 = i * 16, ahead = i + 2 * stride;
    if (i == pos / 16) {
      const int at = pos % 16;
      if (r == at) {
#pragma unroll
        for (int c = 0; c < HD / 16; ++c) t.k[c] = own_k[c];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int key = 4 * g + e;  // what lies behind the step's own key may be no number
#pragma unroll
        for (int c = 0; c < HD / 16; ++c) t.v[c][e] = key == at ? own_v[c] : (key > at ? 0.0f : t.v[c][e]);
      }
    }
    // two chains of products a score, as there
    f32x4 even = {0.0f, 0.0f, 0.0f, 0.0f}, odd = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int c = 0; c < HD / 16; ++c)
#pragma unroll
      for (int j = 0; j < 4; j += 2) {
        even = __builtin_amdgcn_mfma_f32_16x16x4f32(t.k[c][j], q[c][j], even, 0, 0, 0);
        odd = __builtin_amdgcn_mfma_f32_16x16x4f32(t.k[c][j + 1], q[c][j + 1], odd, 0, 0, 0);
      }
    if (ahead < tiles) load_keys(t, ahead);
    f32x4 sc = (even + odd) * a.scale;
#pragma unroll
    for (int e = 0; e < 4; ++e) sc[e] = key0 + 4 * g + e <= pos ? sc[e] : -INFINITY;
    const float top = fmaxf(fmaxf(sc[0], sc[1]), fmaxf(sc[2], sc[3]));
    if (__any(top > reference + kRise)) {
      const float m = fmaxf(most_32_apart(most_16_apart(top)), reference);
      const float factor = reference == -INFINITY ? 0.0f : expf(reference - m);
      reference = m;
      sum *= factor;
#pragma unroll
      for (int c = 0; c < HD / 16; ++c) o[c] *= factor;
    }
    const float against = reference == -INFINITY ? 0.0f : reference;
#pragma unroll
    for (int e = 0; e < 4; ++e) sc[e] = expf(sc[e] - against);
    sum += (sc[0] + sc[1]) + (sc[2] + sc[3]);
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int c = 0; c < HD / 16; ++c) o[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(t.v[c][e], sc[e], o[c], 0, 0, 0);
    if (ahead < tiles) load_values(t, ahead);
    i += stride;
  };
  while (i < tiles) {
    take_tile(one);
    if (i < tiles) take_tile(other);
  }
  sum = sum_32_apart(sum_16_apart(sum));
  if (r < group) {
#pragma unroll
    for (int c = 0; c < HD / 16; ++c) *(f32x4*)&s.attention.o[wave][r][16 * c + 4 * g] = o[c];
  }
  if (g == 0) {
    s.attention.m[wave][r] = reference;
    s.attention.o[wave][r][HD] = sum;
  }
  __syncthreads();
  const Exchange runs(a, a.run_words, a.run_bytes);
  // every wave makes the weights of its states once, a lane a (state, head)
  float (*weights)[kWaves] = s.attention.weights[wave];
  for (int at = lane; at < group * kWaves; at += kWave) {
    const float m = s.attention.m[at % kWaves][at / kWaves];
    float top = m;
    top = fmaxf(top, __shfl_xor(top, 1, kWave));
    top = fmaxf(top, __shfl_xor(top, 2, kWave));
    top = fmaxf(top, __shfl_xor(top, 4, kWave));
    weights[at / kWaves][at % kWaves] = m == -INFINITY ? 0.0f : expf(m - top);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // four channels of a head a thread, and one thread a head for the run's reference and sum
  for (int at = threadIdx.x; at < group * (HD / 4 + 1); at += kWave * kWaves) {
    const int in_group = at / (HD / 4 + 1), four = at % (HD / 4 + 1), of_head = kv_head * group + in_group;
    f32x4 num = {0.0f, 0.0f, 0.0f, 0.0f};
    float den = 0.0f;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const float weight = weights[in_group][w];
      num += *(const f32x4*)&s.attention.o[w][in_group][four < HD / 4 ? 4 * four : 0] * weight;
      den += s.attention.o[w][in_group][HD] * weight;
    }
    float top = s.attention.m[0][in_group];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) top = fmaxf(top, s.attention.m[w][in_group]);
    if (a.splits == 1) {
      num *= 1.0f / den;
      if (four < HD / 4) ex.put(here + a.attn + ((of_head * (HD / 16) + four / 4) * a.m + token) * 16 + four % 4 * 4, marked4(num));
    } else {
      if (four == HD / 4) num = (f32x4){top, den, 0.0f, 0.0f};
      runs.put(layer * a.layer_runs + ((token * a.heads + of_head) * a.splits + split) * kRunRow + 4 * four, marked4(num));
    }
  }
}

// four channels of a (row, head) from its runs, RUNS at once: a head is 16 lanes, a wave has four
template <int RUNS>
__device__ __forceinline__ f32x4 sum_runs(const Exchange& ex, unsigned first_word, int splits, int channel) {
  u32x4 v[RUNS];
  u32x2 state[RUNS];
  ex.take(v, [&](int i) { return At{(first_word + channel) * 4, (unsigned)(i < splits ? i : 0) * kRunRow * 4}; }, state,
          [&](int i) { return At{(first_word + HD) * 4, (unsigned)(i < splits ? i : 0) * kRunRow * 4}; });
  float top = -INFINITY;
#pragma unroll
  for (int i = 0; i < RUNS; ++i) top = i < splits ? fmaxf(top, __uint_as_float(state[i][0])) : top;
  f32x4 num = {0.0f, 0.0f, 0.0f, 0.0f};
  float den = 0.0f;
#pragma unroll
  for (int i = 0; i < RUNS; ++i)
    if (i < splits) {
      const float m = __uint_as_float(state[i][0]), weight = m == -INFINITY ? 0.0f : expf(m - top);
      num += __builtin_bit_cast(f32x4, v[i]) * weight;
      den += __uint_as_float(state[i][1]) * weight;
    }
  return num * (1.0f / den);
}

__device__ __forceinline__ void combine_stage(const ChainArgs32& a, const Exchange& ex, int layer, int block) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int items = a.m * a.heads, first = (block * kWaves + wave) * 4;  // head * rows + row, four a wave
  if (first >= items) return;
  const unsigned here = layer * a.layer_words;
  const int item = min(first + lane / 16, items - 1), head = item / a.m, row = item % a.m, channel = lane % 16 * 4;
  ex.template gate<false>(here + a.q + first * 61 % (items * HD), wave);
  const Exchange runs(a, a.run_words, a.run_bytes);
  const unsigned first_run = layer * a.layer_runs + (row * a.heads + head) * a.splits * kRunRow;
  const f32x4 out = a.splits <= 4 ? sum_runs<4>(runs, first_run, a.splits, channel)
                    : a.splits <= 8 ? sum_runs<8>(runs, first_run, a.splits, channel) : sum_runs<16>(runs, first_run, a.splits, channel);
  ex.put(here + a.attn + ((head * (HD / 16) + channel / 16) * a.m + row) * 16 + channel % 16, marked4(out));
}

template <bool WIDE, int ROWS, bool DOWN>
__device__ __forceinline__ void strip_stage(const ChainArgs32& a, const Exchange& ex, Shared32<ROWS>& s, int layer, int strip) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, r = lane % 16;
  const ChainLayer32& L = a.layers[layer];
  const unsigned here = layer * a.layer_words, next = here + (DOWN ? a.layer_words : 0);
  const int k = DOWN ? a.inner : a.heads * HD;
  const bool last = layer + 1 == a.layer_count;
  constexpr int kSteps = WIDE ? (DOWN ? 32 : 16) : (DOWN ? 12 : 6), kTogether = WIDE ? 8 : 6;
  constexpr int kEach = Ends<ROWS>::kEach;
  Product32<ROWS, 1, kSteps, kTogether, false, false> p;
  p.begin(DOWN ? L.w_down : L.w_o, [&](int) { return strip * 16; }, k, lane, wave);
  const Ends<ROWS> ends(lane);
  const int row = min(ends.row, a.m - 1), column = strip * 16 + ends.first;
  const Floats<kEach> gain = load_floats<kEach>((DOWN ? (last ? L.gain1 : a.layers[layer + 1].gain1) : L.gain2) + column);
  if (WIDE || DOWN) ex.template gate<true>(here + (DOWN ? a.act : a.attn) + strip * 61 % (a.m * k / 16) * 16, wave);
  else if (a.splits > 1) Exchange(a, a.run_words, a.run_bytes).template gate<true>(layer * a.layer_runs + (strip * 61 % (a.m * a.heads * a.splits)) * kRunRow, wave);
  else ex.template gate<true>(here + a.q + strip * 61 % (a.m * a.heads * HD), wave);
  // (the stream is two stages old and more: it is there, and what is looked at before the products is rarely looked for behind them)
  u32x4 held[1];
  auto held_from = [&](int) { return At{(here + (DOWN ? a.plain2 : a.plain1) + (strip * a.m + row) * kRow32 + ends.first / 4 * 4) * 4, 0}; };
  const bool held_there = wave != 0 || ex.template look<kPastCaches>(held, held_from);
  p.run(ex, s, (here + (DOWN ? a.act : a.attn) + min(r, a.m - 1) * 16) * 4, a.m * 64, 0, 0, 0.0f, 0.0f);
  if (!held_there) ex.take(held, held_from);
  Floats<kEach> sums[1];
  float unused;
  if (!p.finish(s, ends, sums, unused, 0.0f)) return;
  if (DOWN && last) {  // (the final norm's kernel adds it to the stream)
    if (ends.row < a.m) {
#pragma unroll
      for (int e = 0; e < kEach; ++e) a.y_out[(size_t)row * a.width + column + e] = sums[0][e];
    }
    return;
  }
  Floats<kEach> v, operand;
  float part = 0.0f;
#pragma unroll
  for (int e = 0; e < kEach; ++e) {
    v[e] = __uint_as_float(kEach == 4 ? held[0][e] : kEach == 2 ? (ends.first % 4 ? held[0][2 + e % 2] : held[0][e]) : held[0][ends.first % 4]) + sums[0][e];
    operand[e] = v[e] * gain[e];
  }
  if constexpr (kEach == 4) {
    part = (v[0] * v[0] + v[kEach - 3] * v[kEach - 3]) + (v[kEach - 2] * v[kEach - 2] + v[kEach - 1] * v[kEach - 1]);
  } else {  // the lane's own, then its neighbours' of the same four channels
    part = kEach == 2 ? v[0] * v[0] + v[kEach - 1] * v[kEach - 1] : v[0] * v[0];
    if constexpr (kEach == 1) part += of_row<0xb1>(part);
    part += of_row<kEach == 1 ? 0x4e : 0xb1>(part);
  }
  part = sum_32_apart(sum_16_apart(part));
  const unsigned to = next + (DOWN ? a.stream1 : a.stream2) + strip * a.strip_words;
  if (ends.first == 0) ex.put(to + a.m * kRow32 + ends.row, marked(part));  // (lanes beyond the rows have the last row's)
  if (ends.row >= a.m) return;
  put_floats(ex, to + row * kRow32 + ends.first, operand);
  put_floats(ex, next + (DOWN ? a.plain1 : a.plain2) + (strip * a.m + row) * kRow32 + ends.first, v);
  if (!DOWN && last) {
#pragma unroll
    for (int e = 0; e < kEach; ++e) a.x_out[(size_t)row * a.width + column + e] = v[e];
  }
}

template <bool WIDE, int ROWS>
__device__ __forceinline__ void gate_stage(const ChainArgs32& a, const Exchange& ex, Shared32<ROWS>& s, int layer, int unit) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, r = lane % 16;
  const ChainLayer32& L = a.layers[layer];
  const unsigned here = layer * a.layer_words;
  constexpr int kSteps = WIDE ? 16 : 6, kTogether = WIDE ? 8 : 6;
  constexpr int kEach = Ends<ROWS>::kEach;
  Product32<ROWS, 2, kSteps, kTogether, true, WIDE> p;
  p.begin(L.w_gate_up, [&](int j) { return j * a.inner + unit * 16; }, a.width, lane, wave);
  const Ends<ROWS> ends(lane);
  const int operand_row = min(r, a.m - 1);
  ex.template gate<true>(a_row(a, here + a.stream2, unit * 61), wave);
  p.run(ex, s, (here + a.stream2 + operand_row * kRow32) * 4, a.strip_words * 4, here + a.stream2 + a.m * kRow32, operand_row, a.inv_width, a.eps);
  Floats<kEach> sums[2], out;
  float scale;
  if (!p.finish(s, ends, sums, scale, a.eps)) return;
  if (ends.row >= a.m) return;
#pragma unroll
  for (int e = 0; e < kEach; ++e) {
    const float gate = sums[0][e] * scale, up = sums[1][e] * scale;
    out[e] = gate / (1.0f + expf(-gate)) * up;
  }
  put_floats(ex, here + a.act + (unit * a.m + ends.row) * 16 + ends.first, out);
}

// Three waves a SIMD: within the 128 registers of four, the attention's two tiles a wave spill 72 of them (batch 8 behind 1,000
// tokens 770 us and not 672).
template <bool WIDE, int ROWS>
__global__ __launch_bounds__(kWave* kWaves) __attribute__((amdgpu_waves_per_eu(WIDE ? 2 : 3))) void chain_f32_kernel(ChainArgs32 a) {
  __shared__ Shared32<ROWS> s;
  const Exchange ex(a, a.words, a.words_bytes, !WIDE);  // (22 layers of width 2,048, 8 rows: 1,427 us and 1,435 with the look through the caches)
  int b = blockIdx.x;
  if (b < a.n_entry) return entry_stage<ROWS>(a, ex, b);
  b -= a.n_entry;
  const int per_layer = a.n_qkv + a.n_att + a.n_comb + 2 * a.n_strip + a.n_gate;
  const int layer = b / per_layer;
  b -= layer * per_layer;
  if (b < a.n_qkv) return qkv_stage<WIDE, ROWS>(a, ex, s, layer, b);
  b -= a.n_qkv;
  if (b < a.n_att) return attention_stage(a, ex, s, layer, b);
  b -= a.n_att;
  if (b < a.n_comb) return combine_stage(a, ex, layer, b);
  b -= a.n_comb;
  if (b < a.n_strip) return strip_stage<WIDE, ROWS, false>(a, ex, s, layer, b);
  b -= a.n_strip;
  if (b < a.n_gate) return gate_stage<WIDE, ROWS>(a, ex, s, layer, b);
  strip_stage<WIDE, ROWS, true>(a, ex, s, layer, b - a.n_gate);
}

// where the words of a layer lie; returns their number
unsigned lay_out(ChainArgs32& a) {
  unsigned at = 0;
  auto place = [&](unsigned& where, unsigned words) {
    where = at;
    at += (words + 31) / 32 * 32;
  };
  const unsigned m = a.m;
  a.strip_words = (kRow32 * m + sum_words(a.width > 1024 ? kMostRows : m) + 15) / 16 * 16;  // (the kernels' ROWS)
  place(a.stream1, a.width / 16 * a.strip_words);
  place(a.stream2, a.width / 16 * a.strip_words);
  place(a.plain1, m * a.width);
  place(a.plain2, m * a.width);
  place(a.q, m * a.heads * HD);
  place(a.k, m * a.kv_heads * HD);
  place(a.v, m * a.kv_heads * HD);
  place(a.attn, m * a.heads * HD);
  place(a.act, m * a.inner);
  a.layer_runs = a.splits > 1 ? m * a.heads * a.splits * kRunRow : 0;
  return at;
}

}  // namespace

// As nnis_chain_words and nnis_chain (chain.hip), with everything in 32 bits: weights [n, k] in the checkpoint's order, y_out in 32
// bits too; up to 16 query heads a key head.
extern "C" long long nnis_chain_f32_words(int layers, int m, int width, int heads, int kv_heads, int inner, int splits, long long* runs) {
  *runs = 0;
  if (layers <= 0 || m < 1 || m > kMostRows || width <= 0 || width % 64 != 0 || width > 8192 || heads <= 0 || kv_heads <= 0 || heads % kv_heads != 0 ||
      heads / kv_heads > 16 || heads * HD > 8192 || inner <= 0 || inner % 64 != 0 || inner > 65536 || splits < 1 || splits > 16) return 0;
  ChainArgs32 a;
  a.m = m; a.width = width; a.heads = heads; a.kv_heads = kv_heads; a.inner = inner; a.splits = splits;
  const long long words = (long long)lay_out(a) * layers + 32;
  *runs = (long long)a.layer_runs * layers;
  return words * 4 < (1LL << 31) && *runs * 4 < (1LL << 31) ? words : 0;
}

extern "C" int nnis_chain_f32(const void* layers, int layer_count, int m, int width, int heads, int kv_heads, int head_dim, int inner, int splits, float eps,
                              float scale, const float* x, float* x_out, float* y_out, const float* tok_cos, const float* tok_sin, const int* tok_pos,
                              const int* tok_page, const int* tok_pages, int max_pages, void* words, long long word_count, void* runs, long long run_count,
                              void* host_fail, void* stream_ptr) {
  long long runs_needed;
  const long long needed = nnis_chain_f32_words(layer_count, m, width, heads, kv_heads, inner, splits, &runs_needed);
  NNIS_REQUIRE(head_dim == HD && needed > 0, "chain_f32: %d rows, width %d, %d/%d heads of %d, inner %d, %d runs are not taken", m, width, heads, kv_heads, head_dim,
               inner, splits);
  NNIS_REQUIRE(layers && x && x_out && y_out && tok_cos && tok_sin && tok_pos && tok_page && tok_pages && max_pages > 0 && words && host_fail,
               "chain_f32: an operand is missing");
  NNIS_REQUIRE(word_count == needed && run_count >= runs_needed && (runs || runs_needed == 0), "chain_f32: %lld and %lld words for %d layers", word_count, run_count,
               layer_count);
  NNIS_REQUIRE(eps > 0.0f && scale > 0.0f, "chain_f32: bad eps or scale");
  for (const void* p : {(const void*)x, (const void*)x_out, (const void*)y_out, (const void*)tok_cos, (const void*)tok_sin, (const void*)words, (const void*)runs})
    NNIS_REQUIRE((uintptr_t)p % 16 == 0, "chain_f32: operands must be 16-byte aligned");
  ChainArgs32 a;
  a.layers = (const ChainLayer32*)layers; a.layer_count = layer_count;
  a.m = m; a.width = width; a.heads = heads; a.kv_heads = kv_heads; a.inner = inner; a.splits = splits;
  a.eps = eps; a.scale = scale; a.inv_width = 1.0f / (float)width;
  a.x = x; a.x_out = x_out; a.y_out = y_out;
  a.tok_cos = tok_cos; a.tok_sin = tok_sin; a.tok_pos = tok_pos; a.tok_page = tok_page; a.tok_pages = tok_pages; a.max_pages = max_pages;
  a.words = (unsigned*)words; a.words_bytes = (unsigned)(word_count * 4);
  a.run_words = (unsigned*)runs; a.run_bytes = (unsigned)(runs_needed * 4);
  a.layer_words = lay_out(a);
  a.fail = a.words + (word_count - 32);
  a.host_fail = (unsigned*)host_fail;
  a.n_strip = width / 16;
  a.n_entry = m;
  a.n_qkv = (heads + 2 * kv_heads) * 2;
  a.n_att = m * kv_heads * splits;
  a.n_comb = splits > 1 ? (m * heads + 4 * kWaves - 1) / (4 * kWaves) : 0;
  a.n_gate = inner / 16;
  const long long blocks = a.n_entry + (long long)layer_count * (a.n_qkv + a.n_att + a.n_comb + 2 * a.n_strip + a.n_gate);
  NNIS_REQUIRE(blocks < (1LL << 30), "chain_f32: too many blocks");
  hipStream_t stream = (hipStream_t)stream_ptr;
  if (chain_clear(words, word_count - 32, runs, runs_needed, a.fail, stream)) return 1;
  if (width > 1024) hipLaunchKernelGGL((chain_f32_kernel<true, 16>), dim3((unsigned)blocks), dim3(kWave * kWaves), 0, stream, a);
  else if (m <= 4) hipLaunchKernelGGL((chain_f32_kernel<false, 4>), dim3((unsigned)blocks), dim3(kWave * kWaves), 0, stream, a);
  else if (m <= 8) hipLaunchKernelGGL((chain_f32_kernel<false, 8>), dim3((unsigned)blocks), dim3(kWave * kWaves), 0, stream, a);
  else hipLaunchKernelGGL((chain_f32_kernel<false, 16>), dim3((unsigned)blocks), dim3(kWave * kWaves), 0, stream, a);
  NNIS_LAUNCH_CHECK("chain_f32");
  return 0;
}
