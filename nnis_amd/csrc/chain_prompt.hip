// The layers of a step of short prompts in one launch: chain.hip's stages for up to 1,024 rows of sequences that begin at their first
// position (pre-norm blocks of plain attention with heads of 64 channels and a SiLU-gated feed-forward, bfloat16).  Where it is
// taken and what it measures there: kernels/ops.py, chain_prompt_takes.
//
// What bounds it is the way from stage to stage, about 3 us of five a layer (30 layers of width 576, 177 rows: 440 of 487 us), and on wide
// models the weights, of which a compute unit holds one block's.
//
// Rows are tiles of 16; a block has a unit of weight rows and 2 or 4 tiles, and 8 waves: K is cut PARTS ways, a wave has a part of K
// and two tiles (four from 65 rows on where the model is wide, for a unit's weights to be read half as often: 128 rows of width 2,048, 22
// layers, 1,503 us and 1,250).  Tiles come in pairs: rows beyond the step's are computed as rows of zeros, so that every word that is
// waited for is written.
//
// Words are handed on as in chain.h.  The blocks of a stage read the same words many times over, and past the caches that would be
// tens of megabytes a stage: the first look through them finds most.  (With a look, past the caches, at a word of each piece before
// it: 177 rows of width 576 536 us and not 482.)  Rows see their own sequence only; its one segment a tile is the usual case
// (segments for all: 495 us and not 487).
#include <hip/hip_runtime.h>

#include "chain.h"
#include "product.h"

namespace {

typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;

constexpr int HD = kChainHead, kWaves = 8;
constexpr int kMostPromptRows = 1024;
constexpr int kPiece = 128;                 // words of 16 rows of a strip of 16 channels in bfloat16
constexpr int kPrepared = 160, kSums = 128; // ... of the stream's, times the next norm's gain: and 16 parts of the rows' sums of squares
constexpr int kPlain = 256;                 // ... in 32 bits
constexpr int kValues = 1024;               // words of 32 keys' values: [channel][8 g + 4 h + e], key 16 h + 4 g + e

struct PromptLayer {
  const bf16_t *w_qkv, *w_o, *w_gate_up, *w_down;  // packed
  const void *gain1, *gain2;
  bf16_t *k_pages, *v_pages;
};

struct PromptArgs {
  const PromptLayer* layers;
  int layer_count, m, tiles, width, heads, kv_heads, inner, gain_dtype;
  float eps, scale_log2, inv_width;
  const float* x;  // [m, width]
  float* x_out;    // [m, width]: the stream behind the last attention
  bf16_t* y_out;   // [m, width]: what the last feed-forward adds to it
  const float *tok_cos, *tok_sin;
  const int *tok_pos, *tok_page;
  unsigned* words;
  unsigned words_bytes, layer_words;
  // where a layer's words lie, all [strip][tile]: the stream before the attention and before the feed-forward, prepared for the
  // product and plain; queries, keys; values [key head][pair of tiles]; attention rows; gated rows
  unsigned ready1, ready2, stream1, stream2, q, k, v, attn, act;
  int n_strip, n_qkv, n_att, n_out, n_gate, n_down;  // blocks of a stage; n_strip: strips of the stream
  unsigned *fail, *host_fail;
};

template <int TILES>
union SharedPrompt {
  struct {
    f32x4 acc[kWaves][TILES][2][kWave];
    float squares[kWaves][TILES][kWave];
  } product;
  struct {
    __attribute__((aligned(16))) float o[kWaves][16][HD + 4];
    float m[kWaves][16], l[kWaves][16];
  } attention;
};

// (unit, group of rows) of a stage's block.  WIDE: the groups of a unit are eight blocks apart, on one die, whose cache then has the unit's
// weights for all but the first; else group by group, as the later ones wait for the earlier ones' keys
template <bool WIDE>
__device__ __forceinline__ void place(int block, int units, int groups, int& unit, int& group) {
  if (!WIDE) {
    unit = block % units;
    group = block / units;
    return;
  }
  const int whole = units / 8 * 8, apart = block < whole * groups ? 8 : units - whole, at = block < whole * groups ? block : block - whole * groups;
  group = at / apart % groups;
  unit = (block < whole * groups ? at / (8 * groups) * 8 : whole) + at % apart;
}

// STRIPS strips of 16 weight rows times the tiles of a block, TILES a wave, K (chunks of 64) cut PARTS ways: part p has the chunks p, p + PARTS, ..
// A wave asks for the weights of its first STEPS chunks when the block begins; TRIP chunks of the operand are asked for together.
template <int STRIPS, int PARTS, int TILES, int STEPS, int TRIP, bool NORM>
struct PromptProduct {
  static constexpr int kBlockTiles = TILES * kWaves / PARTS;
  static_assert(STEPS % TRIP == 0, "whole trips");
  bf16x8 w[STEPS][2][STRIPS];
  f32x4 acc[TILES][STRIPS];
  const bf16_t* strip[STRIPS];
  float square[TILES];
  int chunks, part, wave, lane, tile;

  __device__ __forceinline__ void ask(int base) {
#pragma unroll
    for (int d = 0; d < STEPS; ++d) {
      const int c = base + d * PARTS;
      if (c >= chunks) continue;  // (the same for the whole wave)
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int j = 0; j < STRIPS; ++j) w[d][half][j] = load_chunk(strip[j] + (size_t)c * kPackedChunkElems + half * kPackedHalfElems + lane * 8);
    }
  }
  // row(j): the first weight row of strip j; tile0: the block's first tile
  template <typename Row>
  __device__ __forceinline__ void begin(const bf16_t* weight, Row row, int k, int tile0, int lane_, int wave_) {
    lane = lane_;
    wave = wave_;
    part = wave % PARTS;
    tile = tile0 + wave / PARTS * TILES;
    chunks = nnis_packed_chunks(k);
#pragma unroll
    for (int j = 0; j < STRIPS; ++j) strip[j] = weight + (size_t)(row(j) / 16) * nnis_packed_strip_elems(k);
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
      square[t] = 0.0f;
#pragma unroll
      for (int j = 0; j < STRIPS; ++j) acc[t][j] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    }
    ask(part);
  }
  // the operand [strip][tile] from `words` on, pieces of kPrepared (NORM) or kPiece words
  __device__ __forceinline__ void run(const PromptArgs& a, const Exchange& ex, unsigned words) {
    if (tile >= a.tiles) return;
    constexpr int kWords = NORM ? kPrepared : kPiece;
    const unsigned at = (words + (lane / 16 * a.tiles + tile) * kWords + lane % 16 * 8) * 4;
    for (int base = part; base < chunks; base += PARTS * STEPS) {
      if (base != part) ask(base);
#pragma unroll
      for (int b = 0; b < STEPS; b += TRIP) {
        if (base + b * PARTS >= chunks) continue;
        auto chunk = [&](int d) { return (unsigned)(min(base + (b + d) * PARTS, chunks - 1) * 4 * a.tiles * kWords * 4); };
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
          if (TILES > 2 && tile + t >= a.tiles) continue;
          u32x4 v[TRIP * 2];
          unsigned sums[TRIP];
          auto pieces = [&](int i) { return At{at + i % 2 * 16 + t * kWords * 4, chunk(i / 2)}; };
          if constexpr (NORM) ex.take(v, pieces, sums, [&](int i) { return At{at - lane % 16 * 28 + kSums * 4 + t * kWords * 4, chunk(i)}; });
          else ex.take(v, pieces);
#pragma unroll
          for (int d = 0; d < TRIP; ++d) {
            if (base + (b + d) * PARTS >= chunks) continue;
            if constexpr (NORM) square[t] += __uint_as_float(sums[d]);
#pragma unroll
            for (int half = 0; half < 2; ++half)
#pragma unroll
              for (int j = 0; j < STRIPS; ++j) {
                const bf16x8 x = __builtin_bit_cast(bf16x8, v[d * 2 + half]);
                acc[t][j] = mfma(w[b + d][half][j], x, acc[t][j]);
              }
          }
        }
      }
    }
  }
  // The parts of K added up, a tile a wave; false for waves that have none.  Lane (r, g) gets channels 4 g .. of row r, and that row's
  // scale (NORM).
  __device__ __forceinline__ bool finish(const PromptArgs& a, SharedPrompt<TILES>& s, int tile0, f32x4 (&sums)[STRIPS], float& scale) {
#pragma unroll
    for (int t = 0; t < TILES; ++t) {
#pragma unroll
      for (int j = 0; j < STRIPS; ++j) s.product.acc[wave][t][j][lane] = acc[t][j];
      if constexpr (NORM) s.product.squares[wave][t][lane] = square[t];
    }
    __syncthreads();
    if (wave >= kBlockTiles || tile0 + wave >= a.tiles) return false;
    const int first = wave / TILES * PARTS, t = wave % TILES;
#pragma unroll
    for (int j = 0; j < STRIPS; ++j) {
      sums[j] = s.product.acc[first][t][j][lane];
#pragma unroll
      for (int p = 1; p < PARTS; ++p) sums[j] += s.product.acc[first + p][t][j][lane];
    }
    if constexpr (NORM) {
      float total = s.product.squares[first][t][lane];
#pragma unroll
      for (int p = 1; p < PARTS; ++p) total += s.product.squares[first + p][t][lane];
      scale = 1.0f / sqrtf(sum_32_apart(sum_16_apart(total)) * a.inv_width + a.eps);
    }
    return true;
  }
};

__device__ __forceinline__ u32x2 four_bf16(f32x4 v) {
  return (u32x2){marked2(pack2(v[0], v[1])), marked2(pack2(v[2], v[3]))};
}

__device__ __forceinline__ void entry_stage(const PromptArgs& a, const Exchange& ex, int tile) {
  // (a wave: 16 rows of a strip, four lanes a row)
  for (int i = threadIdx.x; i < a.n_strip * kWave; i += kWaves * kWave) {
    const int strip = i / kWave, r = i % kWave / 4, four = i % 4, row = tile * 16 + r, column = strip * 16 + four * 4;
    f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
    if (row < a.m) v = *(const f32x4*)(a.x + (size_t)row * a.width + column);
    const f32x4 gain = four_of(a.layers[0].gain1, a.gain_dtype, column, 4, true);
    float part = 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) part = fmaf(v[e], v[e], part);
    part += __shfl_xor(part, 1, kWave);
    part += __shfl_xor(part, 2, kWave);
    const unsigned piece = strip * a.tiles + tile;
    ex.put(a.ready1 + piece * kPrepared + r * 8 + four * 2, four_bf16(v * gain));
    if (four == 0) ex.put(a.ready1 + piece * kPrepared + kSums + r, marked(part));
    ex.put(a.stream1 + piece * kPlain + r * 16 + four * 4, (u32x4){marked(v[0]), marked(v[1]), marked(v[2]), marked(v[3])});
  }
}

// queries, keys and values of two strips (a head's channels f .. f + 15 and f + 32 ..), rotated, and the write into the cache
template <bool WIDE, int TILES>
__device__ __forceinline__ void qkv_stage(const PromptArgs& a, const Exchange& ex, SharedPrompt<TILES>& s, int layer, int block) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, r = lane % 16, g = lane / 16;
  const PromptLayer& L = a.layers[layer];
  const unsigned here = layer * a.layer_words;
  typedef PromptProduct<2, WIDE ? 8 : 4, TILES, WIDE ? 4 : 3, WIDE ? 4 : 3, true> P;
  int unit, group;
  place<WIDE>(block, (a.heads + 2 * a.kv_heads) * 2, (a.tiles + P::kBlockTiles - 1) / P::kBlockTiles, unit, group);
  const int tile0 = group * P::kBlockTiles;
  const int head = unit / 2, f0 = unit % 2 * 16;
  P p;
  p.begin(L.w_qkv, [&](int j) { return head * HD + f0 + j * (HD / 2); }, a.width, tile0, lane, wave);
  const int tile = min(tile0 + wave, a.tiles - 1), row = min(tile * 16 + r, a.m - 1);
  const f32x4 c = *(const f32x4*)(a.tok_cos + row * (HD / 2) + f0 + 4 * g), sn = *(const f32x4*)(a.tok_sin + row * (HD / 2) + f0 + 4 * g);
  const int pos = a.tok_pos[row], page = tile * 16 + r < a.m ? a.tok_page[row] : -1;
  ex.template gate<true>(here + a.ready1 + (unit * 61 % a.n_strip * a.tiles + tile0) * kPrepared, wave);
  const bool values = head >= a.heads + a.kv_heads;
  p.run(a, ex, here + a.ready1);
  f32x4 sums[2];
  float scale;
  if (!p.finish(a, s, tile0, sums, scale)) return;
  if (!values) {
    const f32x4 lo = sums[0] * scale, hi = sums[1] * scale;
    const u32x2 out_lo = four_bf16(lo * c - hi * sn), out_hi = four_bf16(hi * c + lo * sn);
    const bool is_key = head >= a.heads;
    const unsigned to = here + (is_key ? a.k : a.q) + (((is_key ? head - a.heads : head) * 4 + f0 / 16) * a.tiles + tile) * kPiece + r * 8 + 2 * g;
    ex.put(to, out_lo);
    ex.put(to + 2 * a.tiles * kPiece, out_hi);
    if (is_key && page >= 0) {
      bf16_t* dst = L.k_pages + ((size_t)page * a.kv_heads + head - a.heads) * nnis_k_page_elems(HD);
      *(u32x2*)(dst + nnis_k_offset(pos % kPageTokens, f0 + 4 * g)) = out_lo;
      *(u32x2*)(dst + nnis_k_offset(pos % kPageTokens, f0 + 4 * g + HD / 2)) = out_hi;
    }
    return;
  }
  // values: lane (r, g) gets the channels f0 + r and f0 + r + 32 of rows 4 g .. 4 g + 3, through what the wave alone reads by now
  const int kv_head = head - a.heads - a.kv_heads, first = wave / TILES * (kWaves / P::kBlockTiles * TILES), t = wave % TILES;
  f32x4(&turn)[2][kWave] = s.product.acc[first][t];
#pragma unroll
  for (int j = 0; j < 2; ++j) turn[j][lane] = sums[j] * scale;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  u32x2 out[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = turn[j][4 * g + e + r / 4 * 16][r % 4];
    out[j] = four_bf16(v);
    ex.put(here + a.v + (kv_head * (a.tiles / 2) + tile / 2) * kValues + 4 * g + tile % 2 * 2 + (f0 + r + j * (HD / 2)) * 16, out[j]);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int to_page = __shfl(page, 4 * g + e, kWave), at = __shfl(pos, 4 * g + e, kWave) % kPageTokens;
    if (to_page < 0) continue;
    unsigned short* dst = (unsigned short*)(L.v_pages + ((size_t)to_page * a.kv_heads + kv_head) * nnis_v_page_elems(HD));
#pragma unroll
    for (int j = 0; j < 2; ++j) dst[nnis_v_offset(f0 + r + j * (HD / 2), at)] = (unsigned short)(out[j][e / 2] >> (e % 2 * 16));
  }
}

// 16 rows of a head against their sequence's keys up to their own, 32 keys a wave: scores as [key][row], whose registers are the
// probabilities' operand in the order of keys that the values have (kValues)
template <int TILES>
__device__ __forceinline__ void attention_stage(const PromptArgs& a, const Exchange& ex, SharedPrompt<TILES>& s, int layer, int block) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, r = lane % 16, g = lane / 16;
  const unsigned here = layer * a.layer_words;
  const int head = block % a.heads, tile = block / a.heads, kv_head = head / (a.heads / a.kv_heads), row = 16 * tile + r;
  const unsigned q = here + a.q + (head * 4 * a.tiles + tile) * kPiece, k = here + a.k + kv_head * 4 * a.tiles * kPiece;
  const unsigned v = here + a.v + kv_head * (a.tiles / 2) * kValues;
  // where the row's sequence begins (padding rows, the last: one from the first of them in the tile on)
  const bool real = row < a.m && a.tok_page[min(row, a.m - 1)] >= 0;
  const int padding = 16 * tile + __popcll(__ballot(real) & 0xffffull);  // (by all lanes)
  const int start = real ? row - a.tok_pos[row] : padding;
  const int first = __builtin_amdgcn_readfirstlane(start);  // (starts do not fall from row to row)
  const bool one = !__any(start != first);
  ex.template gate<true>(q, wave);
  f32x4 o[HD / 16];
#pragma unroll
  for (int c = 0; c < HD / 16; ++c) o[c] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  float reference = -INFINITY, sum = 0.0f;
  for (int pair = first / 32 + wave; pair <= tile / 2; pair += kWaves) {
    u32x4 got[10];
    ex.take(got, [&](int i) {
      if (i < 2) return At{(q + g * a.tiles * kPiece + r * 8 + i * 4) * 4, 0};
      if (i < 6) return At{(k + g * a.tiles * kPiece + r * 8 + i % 2 * 4) * 4, (unsigned)((2 * pair + (i - 2) / 2) * kPiece * 4)};
      return At{(v + r * 16 + g * 4) * 4, (unsigned)(pair * kValues * 4 + (i - 6) * 1024)};
    });
    const int key0 = 32 * pair + 4 * g;  // the lane's eight: key0 + 16 t + e
    f32x4 score[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      score[t] = mfma(__builtin_bit_cast(bf16x8, got[2 + 2 * t]), __builtin_bit_cast(bf16x8, got[0]), (f32x4){0.0f, 0.0f, 0.0f, 0.0f});
      score[t] = mfma(__builtin_bit_cast(bf16x8, got[3 + 2 * t]), __builtin_bit_cast(bf16x8, got[1]), score[t]);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int key = key0 + 16 * t + e;
        score[t][e] = key >= start && key <= row ? score[t][e] * a.scale_log2 : -INFINITY;
      }
    }
    float top = reference;
#pragma unroll
    for (int i = 0; i < 8; ++i) top = fmaxf(top, score[i / 4][i % 4]);
    top = most_32_apart(most_16_apart(top));
    const float base = top == -INFINITY ? 0.0f : top, shrink = __builtin_amdgcn_exp2f(reference - base);
    reference = top;
    sum *= shrink;
    u32x4 p;
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
      const float lo = __builtin_amdgcn_exp2f(score[i / 4][i % 4] - base), hi = __builtin_amdgcn_exp2f(score[i / 4][i % 4 + 1] - base);
      sum += lo;
      sum += hi;
      p[i / 2] = pack2(lo, hi);
    }
#pragma unroll
    for (int c = 0; c < HD / 16; ++c) o[c] *= shrink;
    // A sequence at a time, with the values of no other and for its rows only: what a value is that a row does not see must not
    // matter, and zero times infinity would.
    if (one && 32 * pair >= first) {
#pragma unroll
      for (int c = 0; c < HD / 16; ++c) {
        u32x4 value = got[6 + c];
        if (2 * pair + 1 > tile) value[2] = value[3] = 0;  // (a tile of later rows)
        o[c] = mfma(__builtin_bit_cast(bf16x8, value), __builtin_bit_cast(bf16x8, p), o[c]);
      }
      continue;
    }
    for (int from = first; from >= 0;) {
      int next = start > from ? start : 0x7fffffff;  // the next sequence's first row
#pragma unroll
      for (int offset = 1; offset < 16; offset <<= 1) next = min(next, __shfl_xor(next, offset, kWave));
      const int end = min(next, 16 * tile + 16);
      u32x4 keep;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int key = key0 + 16 * (w / 2) + 2 * (w % 2);
        keep[w] = (key >= from && key < end ? 0xffffu : 0u) | (key + 1 >= from && key + 1 < end ? 0xffff0000u : 0u);
      }
#pragma unroll
      for (int c = 0; c < HD / 16; ++c) {
        const f32x4 with = mfma(__builtin_bit_cast(bf16x8, got[6 + c] & keep), __builtin_bit_cast(bf16x8, p), o[c]);
        o[c] = start == from ? with : o[c];
      }
      from = next < 16 * tile + 16 ? next : -1;
    }
  }
  sum = sum_32_apart(sum_16_apart(sum));
#pragma unroll
  for (int c = 0; c < HD / 16; ++c) *(f32x4*)&s.attention.o[wave][r][16 * c + 4 * g] = o[c];
  if (g == 0) {
    s.attention.m[wave][r] = reference;
    s.attention.l[wave][r] = sum;
  }
  __syncthreads();
  if (wave >= 4) return;
  // wave c: the head's channels 16 c ..; a lane four of them of a row
  const int of_row = lane / 4, four = lane % 4, pairs = tile / 2 + 1 - first / 32;
  float top = -INFINITY, den = 0.0f;
  f32x4 num = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int w = 0; w < kWaves; ++w)
    if (w < pairs) top = fmaxf(top, s.attention.m[w][of_row]);
#pragma unroll
  for (int w = 0; w < kWaves; ++w)
    if (w < pairs) {
      const float m = s.attention.m[w][of_row], weight = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - top);
      num += *(const f32x4*)&s.attention.o[w][of_row][16 * wave + 4 * four] * weight;
      den = fmaf(s.attention.l[w][of_row], weight, den);
    }
  ex.put(here + a.attn + ((head * 4 + wave) * a.tiles + tile) * kPiece + of_row * 8 + four * 2, four_bf16(num * (1.0f / den)));
}

// a strip of 16 columns of the stream: the output projection or the feed-forward's down
template <bool WIDE, int TILES, bool DOWN>
__device__ __forceinline__ void strip_stage(const PromptArgs& a, const Exchange& ex, SharedPrompt<TILES>& s, int layer, int block) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, r = lane % 16, g = lane / 16;
  const PromptLayer& L = a.layers[layer];
  const unsigned here = layer * a.layer_words, next = here + (DOWN ? a.layer_words : 0), from = here + (DOWN ? a.act : a.attn);
  typedef PromptProduct<1, WIDE || DOWN ? 8 : 4, TILES, WIDE ? (DOWN ? 12 : 4) : 3, WIDE ? 4 : 3, false> P;
  int strip, group;
  place<WIDE>(block, a.n_strip, (a.tiles + P::kBlockTiles - 1) / P::kBlockTiles, strip, group);
  const int tile0 = group * P::kBlockTiles, column = strip * 16 + 4 * g;
  const bool last = layer + 1 == a.layer_count;
  P p;
  p.begin(DOWN ? L.w_down : L.w_o, [&](int) { return strip * 16; }, DOWN ? a.inner : a.heads * HD, tile0, lane, wave);
  const f32x4 gain = four_of(DOWN ? (last ? L.gain1 : a.layers[layer + 1].gain1) : L.gain2, a.gain_dtype, column, 4, true);
  ex.template gate<true>(from + (strip * 61 % ((DOWN ? a.inner : a.heads * HD) / 16) * a.tiles + tile0) * kPiece, wave);
  const int tile = min(tile0 + wave, a.tiles - 1), row = tile * 16 + r;
  const unsigned piece = strip * a.tiles + tile;
  u32x4 held[1];
  // (two stages old and more: looked at before the products, and rarely looked for behind them)
  auto held_from = [&](int) { return At{(here + (DOWN ? a.stream2 : a.stream1) + piece * kPlain + r * 16 + 4 * g) * 4, 0}; };
  const bool held_there = wave >= P::kBlockTiles || ex.template look<kPastCaches>(held, held_from);
  p.run(a, ex, from);
  if (!held_there) ex.take(held, held_from);
  f32x4 sums[1];
  float unused;
  if (!p.finish(a, s, tile0, sums, unused)) return;
  if (DOWN && last) {  // (the final norm's kernel adds it to the stream)
    if (row < a.m) {
      bf16x4 y;
#pragma unroll
      for (int e = 0; e < 4; ++e) y[e] = (__bf16)sums[0][e];
      *(bf16x4*)(a.y_out + (size_t)row * a.width + column) = y;
    }
    return;
  }
  f32x4 v;
  float sq = 0.0f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    v[e] = __uint_as_float(held[0][e]) + sums[0][e];
    sq = fmaf(v[e], v[e], sq);
  }
  sq = sum_32_apart(sum_16_apart(sq));
  const unsigned ready = next + (DOWN ? a.ready1 : a.ready2) + piece * kPrepared;
  ex.put(ready + r * 8 + 2 * g, four_bf16(v * gain));
  if (g == 0) ex.put(ready + kSums + r, marked(sq));
  ex.put(next + (DOWN ? a.stream1 : a.stream2) + piece * kPlain + r * 16 + 4 * g, (u32x4){marked(v[0]), marked(v[1]), marked(v[2]), marked(v[3])});
  if (!DOWN && last && row < a.m) *(f32x4*)(a.x_out + (size_t)row * a.width + column) = v;
}

template <bool WIDE, int TILES>
__device__ __forceinline__ void gate_stage(const PromptArgs& a, const Exchange& ex, SharedPrompt<TILES>& s, int layer, int block) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, r = lane % 16, g = lane / 16;
  const unsigned here = layer * a.layer_words;
  typedef PromptProduct<2, WIDE ? 8 : 4, TILES, WIDE ? 4 : 3, WIDE ? 4 : 3, true> P;
  int unit, group;
  place<WIDE>(block, a.inner / 16, (a.tiles + P::kBlockTiles - 1) / P::kBlockTiles, unit, group);
  const int tile0 = group * P::kBlockTiles;
  P p;
  p.begin(a.layers[layer].w_gate_up, [&](int j) { return unit * 16 + j * a.inner; }, a.width, tile0, lane, wave);
  ex.template gate<true>(here + a.ready2 + (unit * 61 % a.n_strip * a.tiles + tile0) * kPrepared, wave);
  p.run(a, ex, here + a.ready2);
  f32x4 sums[2], out;
  float scale;
  if (!p.finish(a, s, tile0, sums, scale)) return;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float gate = sums[0][e] * scale, up = sums[1][e] * scale;
    out[e] = gate * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(gate * -1.4426950408889634f)) * up;  // (as epilogue.h)
  }
  ex.put(here + a.act + (unit * a.tiles + tile0 + wave) * kPiece + r * 8 + 2 * g, four_bf16(out));
}

template <bool WIDE, int TILES>
__global__ __launch_bounds__(kWave* kWaves) __attribute__((amdgpu_waves_per_eu(WIDE ? 2 : 4))) void chain_prompt_kernel(PromptArgs a) {
  __shared__ SharedPrompt<TILES> s;
  const Exchange ex(a, a.words, a.words_bytes);
  int b = blockIdx.x;
  if (b < a.tiles) return entry_stage(a, ex, b);
  b -= a.tiles;
  const int per_layer = a.n_qkv + a.n_att + a.n_out + a.n_gate + a.n_down, layer = b / per_layer;
  b -= layer * per_layer;
  if (b < a.n_qkv) return qkv_stage<WIDE, TILES>(a, ex, s, layer, b);
  b -= a.n_qkv;
  if (b < a.n_att) return attention_stage(a, ex, s, layer, b);
  b -= a.n_att;
  if (b < a.n_out) return strip_stage<WIDE, TILES, false>(a, ex, s, layer, b);
  b -= a.n_out;
  if (b < a.n_gate) return gate_stage<WIDE, TILES>(a, ex, s, layer, b);
  strip_stage<WIDE, TILES, true>(a, ex, s, layer, b - a.n_gate);
}

// where the words of a layer lie; returns their number
long long lay_out(PromptArgs& a) {
  long long at = 0;
  auto place = [&](unsigned& where, long long words) {
    where = (unsigned)at;
    at += words;  // (whole lines: every piece is)
  };
  const long long t = a.tiles, strips = a.width / 16;
  place(a.ready1, strips * t * kPrepared);
  place(a.ready2, strips * t * kPrepared);
  place(a.stream1, strips * t * kPlain);
  place(a.stream2, strips * t * kPlain);
  place(a.q, a.heads * 4 * t * kPiece);
  place(a.k, a.kv_heads * 4 * t * kPiece);
  place(a.v, a.kv_heads * (t / 2) * kValues);
  place(a.attn, a.heads * 4 * t * kPiece);
  place(a.act, a.inner / 16 * t * kPiece);
  return at;
}

}  // namespace

// As nnis_chain_words and nnis_chain (chain.hip), for the m rows of sequences that each begin at their first position and lie one
// behind the other.  Rows with a negative page are computed and not kept; they come last.
extern "C" long long nnis_chain_prompt_words(int layers, int m, int width, int heads, int kv_heads, int inner) {
  if (layers <= 0 || m < 1 || m > kMostPromptRows || width <= 0 || width % 64 != 0 || width > 8192 || heads <= 0 || kv_heads <= 0 || heads % kv_heads != 0 ||
      heads * HD > 8192 || inner <= 0 || inner % 64 != 0 || inner > 65536) return 0;
  PromptArgs a;
  a.tiles = (m + 31) / 32 * 2; a.width = width; a.heads = heads; a.kv_heads = kv_heads; a.inner = inner;
  const long long words = lay_out(a) * layers + 32;
  return words * 4 < (1LL << 31) ? words : 0;
}

extern "C" int nnis_chain_prompt(const void* layers, int layer_count, int m, int width, int heads, int kv_heads, int head_dim, int inner, int gain_dtype, float eps,
                                 float scale, const float* x, float* x_out, void* y_out, const float* tok_cos, const float* tok_sin, const int* tok_pos,
                                 const int* tok_page, void* words, long long word_count, void* host_fail, void* stream_ptr) {
  const long long needed = nnis_chain_prompt_words(layer_count, m, width, heads, kv_heads, inner);
  NNIS_REQUIRE(head_dim == HD && needed > 0, "chain_prompt: %d rows, width %d, %d/%d heads of %d, inner %d are not taken", m, width, heads, kv_heads, head_dim, inner);
  NNIS_REQUIRE(layers && x && x_out && y_out && tok_cos && tok_sin && tok_pos && tok_page && words && host_fail, "chain_prompt: an operand is missing");
  NNIS_REQUIRE(word_count == needed, "chain_prompt: %lld words for %d layers", word_count, layer_count);
  NNIS_REQUIRE(nnis_dtype_ok(gain_dtype) && eps > 0.0f && scale > 0.0f, "chain_prompt: bad gain type, eps or scale");
  for (const void* p : {(const void*)x, (const void*)x_out, (const void*)y_out, (const void*)tok_cos, (const void*)tok_sin, (const void*)words})
    NNIS_REQUIRE((uintptr_t)p % 16 == 0, "chain_prompt: operands must be 16-byte aligned");
  PromptArgs a;
  a.layers = (const PromptLayer*)layers; a.layer_count = layer_count; a.m = m; a.tiles = (m + 31) / 32 * 2;
  a.width = width; a.heads = heads; a.kv_heads = kv_heads; a.inner = inner; a.gain_dtype = gain_dtype;
  a.eps = eps; a.scale_log2 = scale * 1.4426950408889634f; a.inv_width = 1.0f / (float)width;
  a.x = x; a.x_out = x_out; a.y_out = (bf16_t*)y_out; a.tok_cos = tok_cos; a.tok_sin = tok_sin; a.tok_pos = tok_pos; a.tok_page = tok_page;
  a.words = (unsigned*)words; a.words_bytes = (unsigned)(word_count * 4);
  a.layer_words = (unsigned)lay_out(a);
  a.fail = a.words + (word_count - 32);
  a.host_fail = (unsigned*)host_fail;
  const bool wide = width > 1024;
  const bool four = wide && a.tiles > 4;
  const int down = four ? (a.tiles + 3) / 4 : a.tiles / 2, groups = wide ? down : (a.tiles + 3) / 4;  // groups of rows that a block takes
  a.n_strip = width / 16;
  a.n_qkv = (heads + 2 * kv_heads) * 2 * groups;
  a.n_att = heads * a.tiles;
  a.n_out = a.n_strip * groups;
  a.n_gate = inner / 16 * groups;
  a.n_down = a.n_strip * down;
  const long long blocks = a.tiles + (long long)layer_count * (a.n_qkv + a.n_att + a.n_out + a.n_gate + a.n_down);
  NNIS_REQUIRE(blocks < (1LL << 30), "chain_prompt: too many blocks");
  hipStream_t stream = (hipStream_t)stream_ptr;
  if (chain_clear(words, word_count - 32, nullptr, 0, a.fail, stream)) return 1;
  if (four) hipLaunchKernelGGL((chain_prompt_kernel<true, 4>), dim3((unsigned)blocks), dim3(kWave * kWaves), 0, stream, a);
  else if (wide) hipLaunchKernelGGL((chain_prompt_kernel<true, 2>), dim3((unsigned)blocks), dim3(kWave * kWaves), 0, stream, a);
  else hipLaunchKernelGGL((chain_prompt_kernel<false, 2>), dim3((unsigned)blocks), dim3(kWave * kWaves), 0, stream, a);
  NNIS_LAUNCH_CHECK("chain_prompt");
  return 0;
}
