// The layers of a step of few single tokens in one launch (pre-norm blocks of plain attention with heads of 64 channels and a
// SiLU-gated feed-forward, bfloat16, up to 16 rows; up to a width of 1,024 32, as two tiles of rows that have nothing to do with
// one another: 32 rows of 30 layers of width 576 968 us by the layers' kernels; 24 and 32 rows of 100 to 800 tokens 512 and 541 us here; but
// 48 rows of 600 to 2,000 tokens 1,153 and 1,380 when last measured).  How long the sequences may be: kernels/ops.py, chain_longest.
//
// What bounds such a step is neither bytes nor products but its chain of dependent kernels, five to six a layer: each begins
// 1.6 us after the one before has ended, asks for its weights, and only then has something to multiply.  Here a layer's stages
// are blocks of one grid, in the order of the chain: a block asks for its weights (or keys and values) first, waits for its
// operands, and ends with words that the blocks behind it wait for; the chip holds the blocks of two to four layers at a time, so
// a stage's weights are in registers before its operands exist, and from one stage to the next is a store, a load and a
// reduction.
//
// How words get from block to block, and why every wait ends: chain.h.
#include <hip/hip_runtime.h>

#include "chain.h"
#include "product.h"

thread_local char g_nnis_error[512] = {0};
extern "C" const char* nnis_last_error() { return g_nnis_error; }

namespace {

typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;

constexpr int HD = kChainHead, kMostNarrowRows = 32;
constexpr float kLazyRise = 8.0f;  // as in attention.hip: a softmax reference moves when a score rises 2^8 above it

struct ChainLayer {
  const bf16_t *w_qkv, *w_o, *w_gate_up, *w_down;  // packed
  const void *gain1, *gain2;
  bf16_t *k_pages, *v_pages;
};

struct ChainArgs {
  const ChainLayer* layers;
  int layer_count, rows, tiles, m, width, heads, kv_heads, inner, splits, gain_dtype;
  // how many ways K is cut (the first layer's queries, keys and values; the others'; output, gate/up, down), and the waves that
  // share a run's pages
  int parts_first, parts_qkv, parts_out, parts_gate, parts_down, page_waves, down_paired;
  float eps, scale_log2, inv_width;
  const float* x;  // [m, width]
  float* x_out;    // [m, width]: the stream behind the last attention
  bf16_t* y_out;   // [m, width]: what the last feed-forward adds to it
  const float *tok_cos, *tok_sin;
  const int *tok_pos, *tok_page, *tok_pages;
  int max_pages;
  unsigned *words, *run_words;  // (the runs lie apart: in the scratch that the split decode attention has)
  unsigned words_bytes, run_bytes, layer_words, layer_runs;  // of a tile, as m: at most 16 of the step's rows
  // where a layer's words lie: the stream's rows before the attention and before the feed-forward, as operands and in 32 bits; queries,
  // keys, values; attention rows; gated rows
  unsigned stream1, stream2, plain1, plain2, q, k, v, attn, act;
  unsigned strip_words;  // of the stream's rows as the next product takes them
  int n_strip;        // strips of the stream
  int n_qkv, n_att, n_comb, n_out, n_gate, n_down;  // blocks of a stage for a tile (the last may have fewer of the attention's two)
  int n_att_all, n_comb_all;
  int runs_in_out;    // the output projection's blocks add the runs up themselves
  unsigned *fail, *host_fail;
};

// Rows lie by strips of 16 channels: [strip][row][16 bfloat16], 32 bytes that one block writes and that a lane's two pieces of an
// operand are.  A strip of the stream's rows, which is times the next norm's gain, has the rows' parts of their sums of squares
// behind it (a word a row, 4, 8 or 16 of them) and begins on 64 bytes; the stream itself, [strip][row][16], lies apart.  (In one record of 128 bytes a row, every
// piece that a product's block read was a line of its own: a look at 8 rows was 32 lines a load, and the blocks of a stage had their operands
// 1.4 us after the last of them was written: a step of 8 rows, 30 layers of width 576, was 494 us and is 446 with the rows side by side.  Parts of 36 blocks in
// one line took a reader 1.2 us more.)
constexpr int kRowWords = 8;     // of a strip of an operand
constexpr int kPlainWords = 16;  // ... of the stream
// a lane's channels in 16 bits, two a word: four channels are words[0 .. 1], two are words[0]; with one channel a lane words[0] is a word of every other lane,
// whose neighbour has its second half (what the other lanes make is not stored)
template <int N>
__device__ __forceinline__ void pack_row(const Floats<N>& v, unsigned (&words)[2]) {
  if constexpr (N == 1) words[0] = pack2(v[0], of_row<0xb1>(v[0]));
  else words[0] = pack2(v[0], v[1]);
  words[1] = N == 4 ? pack2(v[N == 4 ? 2 : 0], v[N == 4 ? 3 : 0]) : 0;
}
template <int N>
__device__ __forceinline__ void put_packed(const Exchange& ex, unsigned word, int first, const unsigned (&words)[2]) {
  if constexpr (N == 4) ex.put(word + first / 2, (u32x2){marked2(words[0]), marked2(words[1])});
  else if (N == 2 || first % 2 == 0) ex.put(word + first / 2, marked2(words[0]));
}
__device__ __forceinline__ bf16x8 load_packed(const bf16_t* p) { return __builtin_nontemporal_load((const bf16x8*)p); }

// STRIPS strips of 16 weight rows times the step's rows.  K (chunks of 64, whole) is cut `parts` ways: part p has the chunks p, p +
// parts, ..; a wave has V parts, its own number and those WAVES on.  It asks for the weights of its first STEPS chunks when the
// block begins; XB chunks of the operand are asked for together.  A step of the operand beyond the last chunk reads the last again
// and is not multiplied.  The parts and the order of their sums are those of the layers' own kernels for the same product.
// NEXT: a wave's second part is the one after its first, not the one WAVES on.
template <int WAVES, int STRIPS, int STEPS, int XB, int V, bool NEXT = false>
struct Product {
  static_assert(STEPS % XB == 0 && STEPS % V == 0, "whole trips");
  bf16x8 w[STEPS][2][STRIPS];
  f32x4 acc[V][STRIPS];
  const bf16_t* strip[STRIPS];
  int chunks, parts, wave, lane;

  // the chunk of step `s` of the round that begins with a part's chunk number `d0`; `chunks` and more: none
  __device__ __forceinline__ int chunk(int d0, int s) const {
    const int part = NEXT ? V * wave + s / (STEPS / V) : wave + WAVES * (s / (STEPS / V));
    return V > 1 && part >= parts ? chunks : part + parts * (d0 + s % (STEPS / V));
  }
  __device__ __forceinline__ void ask(int d0) {
#pragma unroll
    for (int d = 0; d < STEPS; ++d) {
      const int c = chunk(d0, d);
      if (c >= chunks) continue;  // (the same for the whole wave)
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int j = 0; j < STRIPS; ++j) w[d][half][j] = load_packed(strip[j] + (size_t)c * kPackedChunkElems + half * kPackedHalfElems + lane * 8);
    }
  }
  // row(j): the first row of strip j
  template <typename Row>
  __device__ __forceinline__ void begin(const bf16_t* weight, Row row, int k, int parts_, int lane_, int wave_) {
    parts = parts_;
    wave = wave_;
    lane = lane_;
    chunks = nnis_packed_chunks(k);
#pragma unroll
    for (int j = 0; j < STRIPS; ++j) {
      strip[j] = weight + (size_t)(row(j) / 16) * nnis_packed_strip_elems(k);
#pragma unroll
      for (int v = 0; v < V; ++v) acc[v][j] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
    }
    if (wave < parts) ask(0);
  }
  // the one row from LDS, [step][64], of a K that is one round
  __device__ __forceinline__ void run_row(const bf16x8* row) {
#pragma unroll
    for (int d = 0; d < STEPS; ++d) {
      if (chunk(0, d) >= chunks) continue;
#pragma unroll
      for (int half = 0; half < 2; ++half)
#pragma unroll
        for (int j = 0; j < STRIPS; ++j) acc[0][j] = mfma(w[d][half][j], row[d * 8 + lane / 16 * 2 + half], acc[0][j]);
    }
  }
  // the operand from the exchange: strip s of the lane's row begins at byte `row_at` + s * `stride`; sum(c, part) is called for
  // every chunk with the lane's part of its row's sum of squares, at byte `sum_at` of the strip, if SUM.
  // MORE further loads go with the first trip's, whose offsets `ask_more` gives; `more` has what they brought.
  template <bool SUM, int MORE, typename Sum, typename AskMore>
  __device__ __forceinline__ void run(const Exchange& ex, unsigned row_at, unsigned stride, unsigned sum_at, Sum sum, u32x4 (&more)[MORE > 0 ? MORE : 1], AskMore ask_more) {
    static_assert(!SUM || MORE == 0, "one or the other");
    const unsigned at = row_at + lane / 16 * stride, sums = sum_at + lane / 16 * stride;
    for (int d0 = 0; wave < parts && wave + parts * d0 < chunks; d0 += STEPS / V) {
      if (d0 > 0) ask(d0);
#pragma unroll
      for (int b = 0; b < STEPS; b += XB) {
        if (XB <= STEPS / V && chunk(d0, b) >= chunks) continue;  // (no step of the trip has a chunk)
        u32x4 v[XB * 2 + MORE];
        unsigned part[XB];
        auto step = [&](int d) { return (unsigned)min(chunk(d0, b + d), chunks - 1) * 4 * stride; };
        auto pieces = [&](int i) { return i < XB * 2 ? At{at + i % 2 * 16, step(i / 2)} : ask_more(i - XB * 2); };
        if constexpr (SUM) ex.take(v, pieces, part, [&](int i) { return At{sums, step(i)}; });
        else ex.take(v, pieces);
        if constexpr (MORE > 0) {
#pragma unroll
          for (int i = 0; i < MORE; ++i) more[i] = v[XB * 2 + i];
        }
#pragma unroll
        for (int d = 0; d < XB; ++d) {
          const int c = chunk(d0, b + d);
          if (c >= chunks) continue;
          if constexpr (SUM) sum(c, __uint_as_float(part[d]));
#pragma unroll
          for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int j = 0; j < STRIPS; ++j)
              acc[(b + d) / (STEPS / V)][j] = mfma(w[b + d][half][j], __builtin_bit_cast(bf16x8, v[2 * d + half]), acc[(b + d) / (STEPS / V)][j]);
        }
      }
    }
  }
};

// a word of some row of the stream's strips at `first_word`
__device__ __forceinline__ unsigned a_row(const ChainArgs& a, unsigned first_word, int some) {
  return first_word + some / a.m % a.n_strip * a.strip_words + some % a.m * kRowWords;
}

// units that a block of the products takes: wide models' blocks two, whose rows they then read once
template <int WAVES>
constexpr int units_of() { return WAVES == 8 ? 2 : 1; }

// ... but down's blocks one: a compute unit reads about 30 GB/s, and half as many blocks of twice the weights are late
template <int WAVES, bool DOWN>
constexpr int into_units_of() { return DOWN ? 1 : units_of<WAVES>(); }

template <int WAVES, int ROWS>
struct Shared {
  union {
    struct {
      float acc[WAVES][4][kWave][4];
      float ss[WAVES == 4 ? 1 : WAVES][kWave];  // eight waves: a row's part from each
      RowScales<ROWS> scales;  // four waves
      bf16x8 row[ROWS <= 4 ? WAVES : 1][4 * HD / 8];  // what a wave makes of one row's runs, [step][64]
    } product;
    struct {
      __attribute__((aligned(16))) float o[WAVES][4][HD + 4];  // a head's outputs, then its sum's four parts
      float m[WAVES][4];
      bf16x8 heads[WAVES][kWave];
      __attribute__((aligned(16))) bf16_t stage[WAVES][4][kPageTokens + 8];
    } attention;
    float sums[16];
  };
};

// The parts of K added up, in their order: of a block's UNITS units of NACC strips, unit u's in wave u; false for waves that have none.
template <int WAVES, int ROWS, int UNITS, int NACC, int V>
__device__ __forceinline__ bool add_parts(Shared<WAVES, ROWS>& s, const f32x4 (&acc)[V][UNITS * NACC], Floats<Ends<ROWS>::kEach> (&sums)[NACC], int wave, int lane) {
  constexpr int kEach = Ends<ROWS>::kEach;
  static_assert(V * UNITS * NACC <= 4 && (V == 1 || UNITS == 1), "room for the sums");
#pragma unroll
  for (int v = 0; v < V; ++v)
#pragma unroll
    for (int j = 0; j < UNITS * NACC; ++j) *(f32x4*)s.product.acc[wave][v * UNITS * NACC + j][lane] = acc[v][j];
  const Ends<ROWS> ends(lane);
  __syncthreads();
  if (wave >= UNITS) return false;
#pragma unroll
  for (int j = 0; j < NACC; ++j) {
    auto part_at = [&](int part) { return load_floats<kEach>(&s.product.acc[part % WAVES][part / WAVES * UNITS * NACC + wave * NACC + j][ends.from][ends.first % 4]); };
    sums[j] = part_at(0);
#pragma unroll
    for (int part = 1; part < WAVES * V; ++part) {
      const Floats<kEach> more = part_at(part);
#pragma unroll
      for (int e = 0; e < kEach; ++e) sums[j][e] += more[e];
    }
  }
  return true;
}

// a product with a row that a norm prepared, from the strips at word `first_word`; `sums` and the row's scale in the waves that end a unit
template <int WAVES, int ROWS, int UNITS, int NACC, int V, typename P>
__device__ __forceinline__ bool run_prepared(const ChainArgs& a, const Exchange& ex, Shared<WAVES, ROWS>& s, P& p, unsigned first_word, int row, int wave, int lane,
                                             Floats<Ends<ROWS>::kEach> (&sums)[NACC], float& scale) {
  const unsigned row_at = (first_word + row * kRowWords) * 4, stride = a.strip_words * 4;
  u32x4 none[1];
  // The row's sum of squares is added up as the layers' kernels do: four waves' rows (up to 64 parts) chunk by chunk, all of it by the
  // last wave beside the products; eight waves' each wave's own chunks first.
  if constexpr (WAVES == 4) {
    // (every wave asks for them: with a branch around the products of the one that needs them the kernel keeps 117 registers in scratch memory)
    u32x4 parts[RowScales<ROWS>::kFours];
    auto at = [&](int i) { return RowScales<ROWS>::at(i, lane, first_word + a.m * kRowWords, stride, a.n_strip); };
    p.template run<false, RowScales<ROWS>::kFours>(ex, row_at, stride, 0, [](int, float) {}, parts, at);
    if (wave == WAVES - 1) {
      if (wave >= min(p.parts, p.chunks)) ex.take(parts, at);  // (it had no product)
      s.product.scales.make(parts, lane, a.n_strip, a.inv_width, a.eps);
    }
    if (!add_parts<WAVES, ROWS, UNITS, NACC, V>(s, p.acc, sums, wave, lane)) return false;
    scale = s.product.scales.scale[Ends<ROWS>(lane).row];
    return true;
  }
  float ss = 0.0f;
  p.template run<true, 0>(ex, row_at, stride, (first_word + a.m * kRowWords + row) * 4, [&](int, float part) { ss += part; }, none, [](int) { return At{0, 0}; });
  s.product.ss[wave][lane] = sum_32_apart(sum_16_apart(ss));
  if (!add_parts<WAVES, ROWS, UNITS, NACC, V>(s, p.acc, sums, wave, lane)) return false;
  ss = 0.0f;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) ss += s.product.ss[w][Ends<ROWS>(lane).row];
  scale = 1.0f / sqrtf(ss * a.inv_width + a.eps);
  return true;
}

// The same of eight waves that cut K four ways, waves 0 to 3 for the block's first unit and 4 to 7 for its second.
template <int ROWS, typename P>
__device__ __forceinline__ bool run_prepared_halves(const ChainArgs& a, const Exchange& ex, Shared<8, ROWS>& s, P& p, unsigned first_word, int row, int wave, int lane,
                                                    Floats<Ends<ROWS>::kEach> (&sums)[2], float& scale) {
  constexpr int kEach = Ends<ROWS>::kEach;
  float ss = 0.0f;
  u32x4 none[1];
  p.template run<true, 0>(ex, (first_word + row * kRowWords) * 4, a.strip_words * 4, (first_word + a.m * kRowWords + row) * 4, [&](int, float part) { ss += part; }, none,
                          [](int) { return At{0, 0}; });
  s.product.ss[wave][lane] = sum_32_apart(sum_16_apart(ss));
#pragma unroll
  for (int j = 0; j < 2; ++j) *(f32x4*)s.product.acc[wave][j][lane] = p.acc[0][j];
  const Ends<ROWS> ends(lane);
  __syncthreads();
  if (wave % 4 != 0) return false;
  ss = s.product.ss[wave][ends.row];
#pragma unroll
  for (int w = 1; w < 4; ++w) ss += s.product.ss[wave + w][ends.row];
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    sums[j] = load_floats<kEach>(&s.product.acc[wave][j][ends.from][ends.first % 4]);
#pragma unroll
    for (int w = 1; w < 4; ++w) {
      const Floats<kEach> more = load_floats<kEach>(&s.product.acc[wave + w][j][ends.from][ends.first % 4]);
#pragma unroll
      for (int e = 0; e < kEach; ++e) sums[j][e] += more[e];
    }
  }
  scale = 1.0f / sqrtf(ss * a.inv_width + a.eps);
  return true;
}

// four channels of a row of the embedding: `v`, in 16 bits `operand`, and the strip's part of the sum of squares, the last row's also in place of
// rows that there are none of
template <int ROWS>
__device__ __forceinline__ void put_entry(const ChainArgs& a, const Exchange& ex, int c, int row, f32x4 v, f32x4 operand, float sum) {
  const unsigned strip = c / 16, word = a.stream1 + strip * a.strip_words, four = c % 16 / 4;
  ex.put(word + row * kRowWords + 2 * four, (u32x2){marked2(pack2(operand[0], operand[1])), marked2(pack2(operand[2], operand[3]))});
  ex.put(a.plain1 + (strip * a.m + row) * kPlainWords + 4 * four, (u32x4){marked(v[0]), marked(v[1]), marked(v[2]), marked(v[3])});
  if (four == 0)
    for (int to = row; to < (row + 1 < a.m ? row + 1 : sum_words(ROWS)); ++to) ex.put(word + a.m * kRowWords + to, marked(sum));
}

// A row of the embedding into the first layer's strips.  Of a step of more than 16 rows it is normed as the layers' kernel of its own for
// that does it, a lane per 4 of 256 channels, and its product needs no scale.
template <int ROWS>
__device__ __forceinline__ void normed_entry_stage(const ChainArgs& a, const Exchange& ex, float& shared_scale, int row) {
  const float* x = a.x + (size_t)row * a.width;
  if (threadIdx.x < kWave) {
    float sum = 0.0f;
    for (int c = threadIdx.x * 4; c < a.width; c += kWave * 4) {
      const f32x4 v = *(const f32x4*)(x + c);
#pragma unroll
      for (int e = 0; e < 4; ++e) sum = fmaf(v[e], v[e], sum);
    }
    const float inv_width = 1.0f / (float)a.width, scale = 1.0f / sqrtf(wave_sum(sum) * inv_width + a.eps);
    if (threadIdx.x == 0) shared_scale = scale;
  }
  __syncthreads();
  const float scale = shared_scale;
  for (int c = threadIdx.x * 4; c < a.width; c += blockDim.x * 4) {
    const f32x4 v = *(const f32x4*)(x + c), normed = (v * scale) * four_of(a.layers[0].gain1, a.gain_dtype, c, 4, true);
    put_entry<ROWS>(a, ex, c, row, v, normed, 0.0f);
  }
}

// A row of the embedding into the first layer's strips.  Its sum of squares is one part, added up as the layers' kernel for a row
// that no norm has prepared does: a lane per (part of K, 16 of a chunk's 64 channels).
template <int WAVES, int ROWS>
__device__ __forceinline__ void entry_stage(const ChainArgs& a, const Exchange& ex, Shared<WAVES, ROWS>& s, int row) {
  const float* x = a.x + (size_t)row * a.width;
  if (threadIdx.x < kWave) {
    const int part = threadIdx.x / 4, g = threadIdx.x % 4, parts = a.parts_first;
    float sum = 0.0f;
    for (int c = part; part < parts && c < a.width / 64; c += parts) {
      f32x4 v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = *(const f32x4*)(x + c * 64 + g * 16 + 4 * i);
#pragma unroll
      for (int i = 0; i < 16; ++i) sum = fmaf(v[i / 4][i % 4], v[i / 4][i % 4], sum);
    }
    sum += __shfl_xor(sum, 1, kWave);
    sum += __shfl_xor(sum, 2, kWave);
    float total = __shfl(sum, 0, kWave);
    for (int p = 1; p < parts; ++p) total += __shfl(sum, 4 * p, kWave);
    if (threadIdx.x == 0) s.sums[0] = total;
  }
  __syncthreads();
  const float sum = s.sums[0];
  for (int c = threadIdx.x * 4; c < a.width; c += 64 * WAVES * 4) {
    const f32x4 v = *(const f32x4*)(x + c);
    const f32x4 gain = four_of(a.layers[0].gain1, a.gain_dtype, c, 4, true);
    put_entry<ROWS>(a, ex, c, row, v, v * gain, c == 0 ? sum : 0.0f);
  }
}

// queries, keys and values of two strips (a head's channels f .. f + 15 and f + 32 ..), rotated, and the write into the cache
template <int WAVES, int ROWS, bool FIRST, bool NORMED = false>
__device__ __forceinline__ void qkv_stage(const ChainArgs& a, const Exchange& ex, Shared<WAVES, ROWS>& s, int layer, int unit) {
  constexpr bool kOne = WAVES == 8;
  constexpr int kEach = Ends<ROWS>::kEach;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, r = lane % 16;
  const ChainLayer& L = a.layers[layer];
  const unsigned here = layer * a.layer_words;
  // unit 2 h + i of all: channels 16 i .. 16 i + 15 of head h and those half a head on
  constexpr int kUnits = units_of<WAVES>();
  constexpr int kParts = FIRST && WAVES == 4 ? 2 : 1;  // (a row that no norm has prepared has K cut up to eight ways)
  Product<WAVES, 2 * kUnits, 4, 4, kParts> p;
  p.begin(L.w_qkv, [&](int j) { const int u = unit * kUnits + j / 2; return u / 2 * HD + u % 2 * 16 + j % 2 * (HD / 2); }, a.width,
          FIRST ? a.parts_first : a.parts_qkv, lane, wave);
  const Ends<ROWS> ends(lane);
  const int row = min(ends.row, a.m - 1), unit_here = unit * kUnits + (wave < kUnits ? wave : 0), head = unit_here / 2, f = unit_here % 2 * 16 + ends.first;
  const Floats<kEach> c = load_floats<kEach>(a.tok_cos + row * (HD / 2) + f), sn = load_floats<kEach>(a.tok_sin + row * (HD / 2) + f);
  const int pos = a.tok_pos[row], page = a.tok_page[row];
  ex.template gate<kOne>(a_row(a, here + a.stream1, unit * 61), wave);
  Floats<kEach> sums[2];
  float scale;
  if (!run_prepared<WAVES, ROWS, kUnits, 2, kParts>(a, ex, s, p, here + a.stream1, min(r, a.m - 1), wave, lane, sums, scale)) return;
  if (ends.row >= a.m) return;
  Floats<kEach> out_lo, out_hi;
#pragma unroll
  for (int e = 0; e < kEach; ++e) {
    float lo = sums[0][e] * scale, hi = sums[1][e] * scale;
    if (NORMED && layer == 0) {  // of a normed row, by way of 16 bits, as the layers' two kernels for that
      lo = (float)(__bf16)sums[0][e];
      hi = (float)(__bf16)sums[1][e];
    }
    out_lo[e] = lo;
    out_hi[e] = hi;
    if (head < a.heads + a.kv_heads) {
      out_lo[e] = lo * c[e] - hi * sn[e];
      out_hi[e] = hi * c[e] + lo * sn[e];
    }
  }
  unsigned w_lo[2], w_hi[2];
  pack_row(out_lo, w_lo);
  pack_row(out_hi, w_hi);
  unsigned to;  // [head][strip][row]
  if (head < a.heads) to = a.q + head * a.m * (HD / 2);
  else if (head < a.heads + a.kv_heads) to = a.k + (head - a.heads) * a.m * (HD / 2);
  else to = a.v + (head - a.heads - a.kv_heads) * a.m * (HD / 2);
  to += here + (f / 16 * a.m + row) * 8;
  put_packed<kEach>(ex, to, ends.first, w_lo);
  put_packed<kEach>(ex, to + HD / 32 * a.m * 8, ends.first, w_hi);
  if (page < 0 || head < a.heads) return;
  if (head < a.heads + a.kv_heads) {
    bf16_t* dst = L.k_pages + ((size_t)page * a.kv_heads + head - a.heads) * nnis_k_page_elems(HD);
    unsigned *at_lo = (unsigned*)(dst + nnis_k_offset(pos % kPageTokens, f)), *at_hi = (unsigned*)(dst + nnis_k_offset(pos % kPageTokens, f + HD / 2));
    if constexpr (kEach == 4) {
      *(u32x2*)at_lo = (u32x2){w_lo[0], w_lo[1]};
      *(u32x2*)at_hi = (u32x2){w_hi[0], w_hi[1]};
    } else if (kEach == 2 || f % 2 == 0) {
      *at_lo = w_lo[0];
      *at_hi = w_hi[0];
    }
  } else {
    bf16_t* dst = L.v_pages + ((size_t)page * a.kv_heads + head - a.heads - a.kv_heads) * nnis_v_page_elems(HD);
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
      dst[nnis_v_offset(f + e, pos % kPageTokens)] = (bf16_t)out_lo[e];
      dst[nnis_v_offset(f + HD / 2 + e, pos % kPageTokens)] = (bf16_t)out_hi[e];
    }
  }
}

struct KeysPage {
  bf16x8 k[HD / 8];       // this lane's key, all channels
  bf16x8 v[2][HD / 16];   // value operands of the two halves of the page
};
__device__ __forceinline__ void load_keys(KeysPage& f, const bf16_t* page, int lane) {
#pragma unroll
  for (int c = 0; c < HD / 8; ++c) f.k[c] = *(const bf16x8*)(page + nnis_k_offset(lane, 8 * c));
}
__device__ __forceinline__ void load_values(KeysPage& f, const bf16_t* page, int lane) {
#pragma unroll
  for (int h = 0; h < 2; ++h)
#pragma unroll
    for (int t = 0; t < HD / 16; ++t) f.v[h][t] = *(const bf16x8*)(page + nnis_v_offset(16 * t + lane % 16, 32 * h + 8 * (lane / 16)));
}
__device__ __forceinline__ bf16x4 low4(bf16x8 v) { return __builtin_shufflevector(v, v, 0, 1, 2, 3); }
__device__ __forceinline__ bf16x4 high4(bf16x8 v) { return __builtin_shufflevector(v, v, 4, 5, 6, 7); }

// the largest of a head's lanes: every fourth
__device__ __forceinline__ float top_of_head(float v) {
  v = fmaxf(v, of_row<0x124>(v));
  v = fmaxf(v, of_row<0x128>(v));
  return most_32_apart(most_16_apart(v));
}

// A run of a sequence's keys against up to 4 query heads of a key head, keys on lanes (attention.hip,
// attention_decode_keys_kernel: the same products in the same layouts).  The pages hold every key but the step's own, which the
// projection's blocks of this launch are still writing: it comes from the exchange and takes its place in the page's operands.
template <int WAVES, int ROWS>
__device__ __forceinline__ void attention_stage(const ChainArgs& a, const Exchange& ex, Shared<WAVES, ROWS>& s, int layer, int item) {
  constexpr bool kOne = WAVES == 8;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, r = lane % 16, g = lane / 16;
  const int blk = lane / 4, j = lane % 4;
  const ChainLayer& L = a.layers[layer];
  const unsigned here = layer * a.layer_words;
  const int group = a.heads / a.kv_heads, fours = (group + 3) / 4;
  const int kv_head = item / fours % a.kv_heads, first_head = kv_head * group + item % fours * 4;
  const int token = item / (fours * a.kv_heads) % a.m, split = item / (fours * a.kv_heads * a.m);
  const int heads_here = min(4, kv_head * group + group - first_head);
  const int pos = a.tok_page[token] < 0 ? 0 : a.tok_pos[token];  // a padding row reads its own key only
  const int* pages = a.tok_pages + (size_t)token * a.max_pages;
  const int page_count = pos / kPageTokens + 1;
  const int per_split = (page_count + a.splits - 1) / a.splits;
  const int begin = split * per_split, end = min(begin + per_split, page_count);
  const int first = begin + wave, stride = a.page_waves, mine = wave < stride && end > first ? (end - first + stride - 1) / stride : 0;
  const bf16_t* k_base = L.k_pages + (size_t)kv_head * nnis_k_page_elems(HD);
  const bf16_t* v_base = L.v_pages + (size_t)kv_head * nnis_v_page_elems(HD);
  const size_t k_stride = (size_t)a.kv_heads * nnis_k_page_elems(HD), v_stride = (size_t)a.kv_heads * nnis_v_page_elems(HD);
  KeysPage f;
  if (mine > 0) {
    const size_t page = __builtin_amdgcn_readfirstlane(pages[first]);
    load_keys(f, k_base + page * k_stride, lane);
    load_values(f, v_base + page * v_stride, lane);
  }
  // What lies in a page behind the step's own key may be no number, and zero times that would be none: of the page that a wave
  // has before its operands exist it goes here, where it waits in any case (30 layers of width 576, 1 row: 380 us, all of it below 393,
  // without 385).
  const int own_page = pos / kPageTokens, at_key = pos % kPageTokens;
  auto drop_behind = [&]() {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      u32x4 keep;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int key = 32 * h + 8 * g + 2 * w;
        keep[w] = (key <= at_key ? 0xffffu : 0u) | (key + 1 <= at_key ? 0xffff0000u : 0u);
      }
#pragma unroll
      for (int t = 0; t < HD / 16; ++t) f.v[h][t] = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, f.v[h][t]) & keep);
    }
  };
  if (mine > 0 && first == own_page) drop_behind();
  if (kOne) ex.template gate<kOne>(here + a.q + ((first_head * (HD / 16) + item * 61 % (HD / 16)) * a.m + token) * 8, wave);
  else ex.template gate<kOne>(a_row(a, here + a.stream1, item * 61), wave);
  // Queries and the step's own key and value in one load of the wave (8 lanes a head's row, [head][strip][row]: two pieces a
  // strip), and from there through LDS.
  bf16x8* heads_lds = s.attention.heads[wave];
  {
    const int which = lane / 8, piece = lane % 8;  // 0 to 3: the group's queries; 4, 5: key, value
    const unsigned rows = which < 4 ? a.q + (first_head + (which < heads_here ? which : 0)) * (HD / 2) * a.m : (which == 4 ? a.k : a.v) + kv_head * (HD / 2) * a.m;
    u32x4 v[1];
    ex.take(v, [&](int) { return At{(here + rows + (piece / 2 * a.m + token) * 8 + piece % 2 * 4) * 4, 0}; });
    heads_lds[lane] = which < heads_here || which >= 4 ? __builtin_bit_cast(bf16x8, v[0]) : zero_chunk();
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  bf16x8 q[HD / 8];
#pragma unroll
  for (int c = 0; c < HD / 8; ++c) q[c] = heads_lds[8 * j + c];
  f32x4 o[HD / 16];
#pragma unroll
  for (int t = 0; t < HD / 16; ++t) o[t] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  float reference = -INFINITY, sum = 0.0f;
  bf16_t* stage = &s.attention.stage[wave][0][0];
  constexpr int kStageRow = kPageTokens + 8;
  for (int n = 0; n < mine; ++n) {
    const int index = first + n * stride, key0 = index * kPageTokens;
    if (index == own_page) {  // the step's own key and value take their places in the page's operands
      if (n > 0) drop_behind();
      if (lane == at_key) {
#pragma unroll
        for (int c = 0; c < HD / 8; ++c) f.k[c] = heads_lds[32 + c];
      }
      // (the word that the key's value is half of is the same in all lanes: a branch a word, not a choice a register)
      const int word_at = __builtin_amdgcn_readfirstlane(at_key / 32 * 4 + at_key % 8 / 2), of_lanes = at_key % 32 / 8;
      const unsigned keep = at_key % 2 ? 0xffffu : 0xffff0000u, shift = at_key % 2 * 16;
      const unsigned short* value = (const unsigned short*)(heads_lds + 40) + r;
      unsigned channel[HD / 16];
#pragma unroll
      for (int t = 0; t < HD / 16; ++t) channel[t] = (unsigned)value[16 * t] << shift;
#pragma unroll
      for (int w = 0; w < 8; ++w) {
        if (w != word_at) continue;
        asm volatile("");  // (a branch)
#pragma unroll
        for (int t = 0; t < HD / 16; ++t) {
          u32x4 words = __builtin_bit_cast(u32x4, f.v[w / 4][t]);
          words[w % 4] = g == of_lanes ? (words[w % 4] & keep) | channel[t] : words[w % 4];
          f.v[w / 4][t] = __builtin_bit_cast(bf16x8, words);
        }
      }
    }
    f32x4 s0 = {0.0f, 0.0f, 0.0f, 0.0f}, s1 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int c = 0; c < HD / 8; ++c) {
      s0 = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(low4(f.k[c]), low4(q[c]), s0, 0, 0, 0);
      s1 = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(high4(f.k[c]), high4(q[c]), s1, 0, 0, 0);
    }
    const bool more = n + 1 < mine;
    const size_t next = more ? __builtin_amdgcn_readfirstlane(pages[index + stride]) : 0;
    if (more) load_keys(f, k_base + next * k_stride, lane);
    f32x4 sc = s0 + s1;
    float top = -INFINITY;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      sc[e] = key0 + 4 * blk + e <= pos ? sc[e] * a.scale_log2 : -INFINITY;
      top = fmaxf(top, sc[e]);
    }
    if (__any(top > reference + kLazyRise)) {
      const float moved = top_of_head(fmaxf(reference, top));
      const float shrink = reference == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(reference - moved);
      sum *= shrink;
#pragma unroll
      for (int t = 0; t < HD / 16; ++t) o[t] = o[t] * shrink;
      reference = moved;
    }
    const float base = reference == -INFINITY ? 0.0f : reference;
    bf16x4 p;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float w = __builtin_amdgcn_exp2f(sc[e] - base);
      sum += w;
      p[e] = (__bf16)w;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    *(bf16x4*)(stage + j * kStageRow + 4 * blk) = p;
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      bf16x8 columns = *(const bf16x8*)(stage + (r < 4 ? r : 0) * kStageRow + 32 * h + 8 * g);
      if (r >= 4) columns = zero_chunk();
#pragma unroll
      for (int t = 0; t < HD / 16; ++t) o[t] = mfma(f.v[h][t], columns, o[t]);
    }
    if (more) load_values(f, v_base + next * v_stride, lane);
  }
  // the states meet in LDS: a lane group's part of a head's sum is that of the keys 16 g .. 16 g + 15 of its pages
  sum += of_row<0x12c>(sum);  // (four lanes on; right in the four lanes that are stored)
  sum += of_row<0x128>(sum);
  if (r < 4) {
#pragma unroll
    for (int t = 0; t < HD / 16; ++t) *(f32x4*)&s.attention.o[wave][r][16 * t + 4 * g] = o[t];
    s.attention.o[wave][r][HD + g] = sum;
    if (g == 0) s.attention.m[wave][r] = reference;
  }
  __syncthreads();
  const Exchange runs(a, a.run_words, a.run_bytes);
  // four channels of a head a thread, and one thread a head for the run's reference and sum
  for (int i = threadIdx.x; i < heads_here * (HD / 4 + 1); i += 64 * WAVES) {
    const int head = i / (HD / 4 + 1), four = i % (HD / 4 + 1);
    // the waves' states in halving rounds, as the layers' kernel has them; the one thread's four are the sum's parts
    float m[WAVES];
    f32x4 out[WAVES], l[WAVES];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      m[w] = s.attention.m[w][head];
      out[w] = *(const f32x4*)&s.attention.o[w][head][4 * four];
      if (a.splits == 1) l[w] = *(const f32x4*)&s.attention.o[w][head][HD];
    }
#pragma unroll
    for (int half = WAVES / 2; half >= 1; half >>= 1) {
      if (half >= a.page_waves) continue;
#pragma unroll
      for (int w = 0; w < half; ++w) {
        const float m_new = fmaxf(m[w], m[w + half]), m_safe = m_new == -INFINITY ? 0.0f : m_new;
        const float mine_w = __builtin_amdgcn_exp2f(m[w] - m_safe), their_w = __builtin_amdgcn_exp2f(m[w + half] - m_safe);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          // (which of a sum's two products is rounded first is the compiler's choice there: the other one for the last 16 channels)
          const bool other = four >= 12 && four < HD / 4;
          const float first = other ? out[w][e] : out[w + half][e], second = other ? out[w + half][e] : out[w][e];
          out[w][e] = fmaf(first, other ? mine_w : their_w, second * (other ? their_w : mine_w));
          if (a.splits == 1) l[w][e] = fmaf(l[w + half][e], their_w, l[w][e] * mine_w);
        }
        m[w] = m_new;
      }
    }
    f32x4 num = out[0];
    if (a.splits == 1) {
      const float inv = 1.0f / ((l[0][0] + l[0][1]) + (l[0][2] + l[0][3]));
#pragma unroll
      for (int e = 0; e < 4; ++e) num[e] = num[e] * inv;
      if (four < HD / 4)
        ex.put(here + a.attn + (((first_head + head) * (HD / 16) + four / 4) * a.m + token) * 8 + four % 4 * 2,
               (u32x2){marked2((bf16_t)num[0], (bf16_t)num[1]), marked2((bf16_t)num[2], (bf16_t)num[3])});
    } else {
      if (four == HD / 4) num = (f32x4){m[0], (num[0] + num[1]) + (num[2] + num[3]), 0.0f, 0.0f};
      runs.put(layer * a.layer_runs + ((token * a.heads + first_head + head) * a.splits + split) * kRunRow + 4 * four,
             (u32x4){marked(num[0]), marked(num[1]), marked(num[2]), marked(num[3])});
    }
  }
}

__device__ __forceinline__ float rounded_sum(float sum, float a, float b) {
#pragma clang fp contract(off)
  const float product = a * b;
  return sum + product;
}

// Four channels of a (row, head) from its runs, RUNS at once: a head is 16 lanes, a wave has four.  alone: in the roundings of the
// layers' kernel of its own for this sum, not of the output projection that makes it on the way (up to four rows, of up to 2,040
// channels: 16 rows of them in its LDS; nnis_gemm_residual_runs_fits).
template <int RUNS>
__device__ __forceinline__ bf16x4 sum_runs(const Exchange& ex, unsigned first_word, int splits, int channel, bool alone) {
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
      const float m = __uint_as_float(state[i][0]), weight = m == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m - top);
      num += __builtin_bit_cast(f32x4, v[i]) * weight;
      const float add = __uint_as_float(state[i][1]);
      den = alone ? rounded_sum(den, add, weight) : fmaf(add, weight, den);
    }
  bf16x4 out;
#pragma unroll
  for (int e = 0; e < 4; ++e) out[e] = (__bf16)(num[e] / den);
  return out;
}
template <int WAVES>
__device__ __forceinline__ void combine_stage(const ChainArgs& a, const Exchange& ex, int layer, int block) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int items = a.m * a.heads, first = (block * WAVES + wave) * 4;  // head * rows + row, four a wave: whole lines of the rows' strips
  if (first >= items) return;
  const unsigned here = layer * a.layer_words;
  const int item = min(first + lane / 16, items - 1), head = item / a.m, row = item % a.m, channel = lane % 16 * 4;
  ex.template gate<false>(here + a.q + first * 61 % (items * (HD / 2)), 0);
  const Exchange runs(a, a.run_words, a.run_bytes);
  const bool alone = a.rows > 4 || a.heads * HD > 2040;
  const unsigned first_run = layer * a.layer_runs + (row * a.heads + head) * a.splits * kRunRow;
  const bf16x4 out = a.splits <= 4 ? sum_runs<4>(runs, first_run, a.splits, channel, alone)
                     : a.splits <= 8 ? sum_runs<8>(runs, first_run, a.splits, channel, alone) : sum_runs<16>(runs, first_run, a.splits, channel, alone);
  ex.put(here + a.attn + ((head * (HD / 16) + channel / 16) * a.m + row) * 8 + channel % 16 / 2,
         (u32x2){marked2(out[0], out[1]), marked2(out[2], out[3])});
}

// a strip of 16 columns of the stream: the output projection (down = false) or the feed-forward's down
// PAIRED: K cut sixteen ways, the even parts and the odd ones added up apart, as the layers' kernel does in two blocks
template <int WAVES, int ROWS, bool DOWN, bool PAIRED>
__device__ __forceinline__ void strip_stage(const ChainArgs& a, const Exchange& ex, Shared<WAVES, ROWS>& s, int layer, int block) {
  constexpr bool kOne = WAVES == 8;
  constexpr int kEach = Ends<ROWS>::kEach;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, r = lane % 16;
  const ChainLayer& L = a.layers[layer];
  const unsigned here = layer * a.layer_words, next = here + (DOWN ? a.layer_words : 0);
  const int k = DOWN ? a.inner : a.heads * HD;
  const bool last = DOWN && layer + 1 == a.layer_count;
  // a wave's steps whose weights are in registers before the operands exist: 4 waves have 6 of an inner size of 1,536, 8 waves 11 of 5,632
  constexpr int kUnits = into_units_of<WAVES, DOWN>(), kSteps = WAVES == 4 ? (DOWN ? 6 : 4) : (DOWN ? 16 : 4), kTogether = WAVES == 4 ? kSteps : 4;
  constexpr int kParts = (WAVES == 4 && DOWN) || PAIRED ? 2 : 1;
  Product<WAVES, kUnits, kSteps, kTogether, kParts, PAIRED> p;
  p.begin(DOWN ? L.w_down : L.w_o, [&](int j) { return (block * kUnits + j) * 16; }, k, PAIRED ? 16 : DOWN ? a.parts_down : a.parts_out, lane, wave);
  const Ends<ROWS> ends(lane);
  const int strip = block * kUnits + (wave < kUnits ? wave : 0), row = min(ends.row, a.m - 1), column = strip * 16 + ends.first;
  const void* gain_of = DOWN ? (last ? L.gain1 : a.layers[layer + 1].gain1) : L.gain2;
  const f32x4 gains = four_of(gain_of, a.gain_dtype, column / 4 * 4, 4, true);
  Floats<kEach> gain;
#pragma unroll
  for (int e = 0; e < kEach; ++e) gain[e] = kEach == 4 ? gains[e] : kEach == 2 ? (ends.first % 4 ? gains[2 + e % 2] : gains[e]) : gains[ends.first % 4];
  if (DOWN || (kOne && !(ROWS <= 4 && a.runs_in_out))) ex.template gate<kOne>(here + (DOWN ? a.act : a.attn) + block * 61 % (a.m * k / 16) * 8, wave);
  else if (a.splits > 1) Exchange(a, a.run_words, a.run_bytes).template gate<kOne>(layer * a.layer_runs + (block * 61 % (a.m * a.heads * a.splits)) * kRunRow, wave);
  else ex.template gate<kOne>(here + a.q + block * 61 % (a.m * a.heads * (HD / 2)), wave);
  // (the stream is two stages old and more: it is there, and what is looked at before the products is rarely looked for behind them)
  const unsigned held_at = here + (DOWN ? a.plain2 : a.plain1) + (strip * a.m + row) * kPlainWords + ends.first / 4 * 4;
  u32x4 held[1], none[1];
  auto held_from = [&](int) { return At{held_at * 4, 0}; };
  const bool held_there = wave >= kUnits || ex.template look<kPastCaches>(held, held_from);
  bool from_runs = false;
  if constexpr (!DOWN && ROWS <= 4) {
    from_runs = a.runs_in_out;
    if (from_runs && wave < min(p.parts, p.chunks)) {
      // One row: a head is a step of K, and 16 lanes of the wave that multiplies it add its runs up (an exchange less: 30 layers of width
      // 576 behind 700 keys 370 -> 347 us, behind 3,000 in eight runs 403 -> 383; of 2 rows 378 and 380, of 4 382 and 433).
      const Exchange runs(a, a.run_words, a.run_bytes);
      const int head = min(p.chunk(0, lane / 16), p.chunks - 1), channel = lane % 16 * 4;
      const unsigned first_run = layer * a.layer_runs + head * a.splits * kRunRow;
      const bool alone = WAVES == 8 && a.heads * HD > 2040;  // (as combine_stage)
      ((bf16x4*)s.product.row[wave])[lane] = a.splits <= 4 ? sum_runs<4>(runs, first_run, a.splits, channel, alone) : sum_runs<8>(runs, first_run, a.splits, channel, alone);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      p.run_row(s.product.row[wave]);
    }
  }
  if (!from_runs)
    p.template run<false, 0>(ex, (here + (DOWN ? a.act : a.attn) + min(r, a.m - 1) * 8) * 4, a.m * 32, 0, [](int, float) {}, none, [](int) { return At{0, 0}; });
  if (!held_there) ex.take(held, held_from);
  Floats<kEach> sums[1];
  if constexpr (PAIRED) {
    const f32x4 even[1][1] = {{p.acc[0][0]}};
    *(f32x4*)s.product.acc[wave][1][lane] = p.acc[1][0];
    if (!add_parts<WAVES, ROWS, 1, 1, 1>(s, even, sums, wave, lane)) return;
    auto odd_at = [&](int w) { return load_floats<kEach>(&s.product.acc[w][1][ends.from][ends.first % 4]); };
    Floats<kEach> odd = odd_at(0);
#pragma unroll
    for (int w = 1; w < WAVES; ++w) {
      const Floats<kEach> more = odd_at(w);
#pragma unroll
      for (int e = 0; e < kEach; ++e) odd[e] += more[e];
    }
#pragma unroll
    for (int e = 0; e < kEach; ++e) sums[0][e] += odd[e];
  } else {
    if (!add_parts<WAVES, ROWS, kUnits, 1, kParts>(s, p.acc, sums, wave, lane)) return;
  }
  if (last) {  // (the final norm's kernel adds it to the stream)
    if (ends.row < a.m) {
#pragma unroll
      for (int e = 0; e < kEach; ++e) a.y_out[(size_t)row * a.width + column + e] = (bf16_t)sums[0][e];
    }
    return;
  }
  Floats<kEach> v, operand;
#pragma unroll
  for (int e = 0; e < kEach; ++e) {
    v[e] = __uint_as_float(kEach == 4 ? held[0][e] : kEach == 2 ? (ends.first % 4 ? held[0][2 + e % 2] : held[0][e]) : held[0][ends.first % 4]) + sums[0][e];
    operand[e] = v[e] * gain[e];
  }
  unsigned words[2];
  pack_row(operand, words);
  // a lane group's four channels in their order
  float sq = 0.0f;
  if constexpr (kEach == 1) {
    const float v0 = of_row<0x00>(v[0]), v1 = of_row<0x55>(v[0]), v2 = of_row<0xaa>(v[0]), v3 = of_row<0xff>(v[0]);
    sq = fmaf(v3, v3, fmaf(v2, v2, fmaf(v1, v1, fmaf(v0, v0, 0.0f))));
  } else if constexpr (kEach == 2) {
    const float v0 = of_row<0xa0>(v[0]), v1 = of_row<0xa0>(v[1]), v2 = of_row<0xf5>(v[0]), v3 = of_row<0xf5>(v[1]);
    sq = fmaf(v3, v3, fmaf(v2, v2, fmaf(v1, v1, fmaf(v0, v0, 0.0f))));
  } else {
#pragma unroll
    for (int e = 0; e < kEach; ++e) sq = fmaf(v[e], v[e], sq);
  }
  sq = sum_32_apart(sum_16_apart(sq));
  const unsigned to = next + (DOWN ? a.stream1 : a.stream2) + strip * a.strip_words;
  if (ends.first == 0) ex.put(to + a.m * kRowWords + ends.row, marked(sq));  // (lanes beyond the rows have the last row's)
  if (ends.row >= a.m) return;
  put_packed<kEach>(ex, to + row * kRowWords, ends.first, words);
  put_floats(ex, next + (DOWN ? a.plain1 : a.plain2) + (strip * a.m + row) * kPlainWords + ends.first, v);
  if (!DOWN && layer + 1 == a.layer_count) {
#pragma unroll
    for (int e = 0; e < kEach; ++e) a.x_out[(size_t)row * a.width + column + e] = v[e];
  }
}

// HALVES: eight waves that cut K four ways for each of the block's two units, as the layers' kernel does for this many strips
template <int WAVES, int ROWS, bool HALVES>
__device__ __forceinline__ void gate_stage(const ChainArgs& a, const Exchange& ex, Shared<WAVES, ROWS>& s, int layer, int block) {
  constexpr bool kOne = WAVES == 8;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave, r = lane % 16;
  const unsigned here = layer * a.layer_words;
  constexpr int kUnits = units_of<WAVES>();
  const int unit = block * kUnits + (HALVES ? wave / 4 : wave < kUnits ? wave : 0), row = min(r, a.m - 1);
  const unsigned one = a_row(a, here + a.stream2, block * 61);
  constexpr int kEach = Ends<ROWS>::kEach;
  const Ends<ROWS> ends(lane);
  Floats<kEach> sums[2];
  float scale;
  if constexpr (HALVES) {
    Product<4, 2, 8, 4, 1> p;
    p.begin(a.layers[layer].w_gate_up, [&](int j) { return unit * 16 + j * a.inner; }, a.width, 4, lane, wave % 4);
    ex.template gate<kOne>(one, wave);
    if (!run_prepared_halves(a, ex, s, p, here + a.stream2, row, wave, lane, sums, scale)) return;
  } else {
    Product<WAVES, 2 * kUnits, 4, 4, 1> p;
    p.begin(a.layers[layer].w_gate_up, [&](int j) { return (block * kUnits + j / 2) * 16 + j % 2 * a.inner; }, a.width, a.parts_gate, lane, wave);
    ex.template gate<kOne>(one, wave);
    if (!run_prepared<WAVES, ROWS, kUnits, 2, 1>(a, ex, s, p, here + a.stream2, row, wave, lane, sums, scale)) return;
  }
  if (ends.row >= a.m) return;
  Floats<kEach> out;
#pragma unroll
  for (int e = 0; e < kEach; ++e) {
    const float gate = sums[0][e] * scale, up = sums[1][e] * scale;
    const float x = __builtin_amdgcn_exp2f(gate * -1.4426950408889634f);  // (as epilogue.h)
    out[e] = gate * __builtin_amdgcn_rcpf(1.0f + x) * up;
  }
  unsigned words[2];
  pack_row(out, words);
  put_packed<kEach>(ex, here + a.act + (unit * a.m + ends.row) * 8, ends.first, words);
}

// TILED: more than 16 rows (beside its arithmetic steps of up to 16 are half a per cent slower).  NEAR: the first look through the caches
// (Exchange::take): it needs registers that fewer than five rows lose more by than they gain (four waves, of 30 layers of width 576, without
// and with it: 1 row 387 and 391 us, 4 458 and 462, 8 491 and 480, 16 566 and 550, 17 643 and 603).
template <int WAVES, int ROWS, bool TILED, bool NEAR>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(WAVES == 4 && (TILED || !NEAR) ? 3 : 2))) void chain_kernel(ChainArgs a) {
  __shared__ Shared<WAVES, ROWS> s;
  int b = blockIdx.x, layer = -1, stage = -1, tile = 0;
  auto in = [&](int index, int blocks, int all) {  // the stage with this index has `blocks` for a tile
    if (stage >= 0) return;
    if (b < all) {
      stage = index;
      if (TILED) {
        tile = b / blocks;
        b -= tile * blocks;
      }
    } else {
      b -= all;
    }
  };
  in(0, kMostRows, a.rows);
  if (stage < 0) {
    const int per_layer = a.tiles * (a.n_qkv + a.n_out + a.n_gate + a.n_down) + a.n_att_all + a.n_comb_all;
    layer = b / per_layer;
    b -= layer * per_layer;
    in(1, a.n_qkv, a.tiles * a.n_qkv);
    in(2, a.n_att, a.n_att_all);
    in(3, a.n_comb, a.n_comb_all);
    in(4, a.n_out, a.tiles * a.n_out);
    in(5, a.n_gate, a.tiles * a.n_gate);
    in(6, a.n_down, a.tiles * a.n_down);
  }
  if constexpr (TILED) {  // from here on the tile's rows are all there is
    a.x += (size_t)tile * kMostRows * a.width;
    a.x_out += (size_t)tile * kMostRows * a.width;
    a.y_out += (size_t)tile * kMostRows * a.width;
    a.tok_cos += tile * kMostRows * (HD / 2);
    a.tok_sin += tile * kMostRows * (HD / 2);
    a.tok_pos += tile * kMostRows;
    a.tok_page += tile * kMostRows;
    a.tok_pages += (size_t)tile * kMostRows * a.max_pages;
    a.words += (size_t)tile * a.layer_count * a.layer_words;
    a.run_words += (size_t)tile * a.layer_count * a.layer_runs;
    a.m = min(kMostRows, a.rows - tile * kMostRows);
  }
  const Exchange ex(a, a.words, a.words_bytes, NEAR);
  if (stage == 0) {
    if (TILED) return normed_entry_stage<ROWS>(a, ex, s.sums[0], b);
    return entry_stage<WAVES, ROWS>(a, ex, s, b);
  }
  if (stage == 1) {
    if (WAVES == 4 && !TILED && layer == 0) return qkv_stage<WAVES, ROWS, true>(a, ex, s, layer, b);
    return qkv_stage<WAVES, ROWS, false, TILED>(a, ex, s, layer, b);
  }
  if (stage == 2) return attention_stage<WAVES, ROWS>(a, ex, s, layer, b);
  if (stage == 3) return combine_stage<WAVES>(a, ex, layer, b);
  if (stage == 4) return strip_stage<WAVES, ROWS, false, false>(a, ex, s, layer, b);
  if (stage == 5) {
    if constexpr (WAVES == 8)
      if (a.parts_gate == 4) return gate_stage<WAVES, ROWS, true>(a, ex, s, layer, b);
    return gate_stage<WAVES, ROWS, false>(a, ex, s, layer, b);
  }
  if constexpr (WAVES == 8)
    if (a.down_paired && layer + 1 < a.layer_count) return strip_stage<WAVES, ROWS, true, true>(a, ex, s, layer, b);
  strip_stage<WAVES, ROWS, true, false>(a, ex, s, layer, b);
}

// where the words of a layer lie; returns their number
unsigned lay_out(ChainArgs& a) {
  unsigned at = 0;
  auto place = [&](unsigned& where, unsigned words) {
    where = at;
    at += (words + 31) / 32 * 32;
  };
  const unsigned m = a.m, strips = a.width / 16;
  a.strip_words = (kRowWords * m + sum_words(a.width > 1024 && m > 4 ? kMostRows : m) + 15) / 16 * 16;  // (the kernels' ROWS)
  place(a.stream1, strips * a.strip_words);
  place(a.stream2, strips * a.strip_words);
  place(a.plain1, m * strips * kPlainWords);
  place(a.plain2, m * strips * kPlainWords);
  place(a.q, m * a.heads * (HD / 2));
  place(a.k, m * a.kv_heads * (HD / 2));
  place(a.v, m * a.kv_heads * (HD / 2));
  place(a.attn, m * a.heads * (HD / 2));
  place(a.act, m * a.inner / 2);
  a.layer_runs = a.splits > 1 ? m * a.heads * a.splits * kRunRow : 0;
  return at;
}

bool fits(int m, int width, int heads, int kv_heads, int inner, int splits) {
  return m >= 1 && m <= (width > 1024 ? kMostRows : kMostNarrowRows) && width > 0 && width % 64 == 0 && width <= 8192 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0 && heads * HD <= 8192 &&
         inner > 0 && inner % 64 == 0 && inner <= 65536 && splits >= 1 && splits <= 16;
}

}  // namespace

// Words that a step's exchange needs (of 4 bytes; the last 32 are the kernel's own), or 0 for sizes that it does not take; `runs`: the
// words of the runs beside them.
extern "C" long long nnis_chain_words(int layers, int m, int width, int heads, int kv_heads, int inner, int splits, long long* runs) {
  *runs = 0;
  if (layers <= 0 || !fits(m, width, heads, kv_heads, inner, splits)) return 0;
  ChainArgs a;
  const int tiles = (m + kMostRows - 1) / kMostRows;
  a.m = min(m, kMostRows); a.width = width; a.heads = heads; a.kv_heads = kv_heads; a.inner = inner; a.splits = splits;
  const long long words = (long long)lay_out(a) * layers * tiles + 32;
  *runs = (long long)a.layer_runs * layers * tiles;
  return words * 4 < (1LL << 31) && *runs * 4 < (1LL << 31) ? words : 0;
}

// The layers of one step of single tokens.  layers: device memory, 8 pointers a layer (packed weights of q/k/v, output, gate/up
// and down; the gains of its two norms, all of gain_dtype; its key and value pages); x, x_out: [m, width] in 32 bits; tok_cos,
// tok_sin, tok_page, tok_pages: the step's tables.  words, runs: as nnis_chain_words says, 16-byte aligned.  host_fail: a word of pinned
// host memory.
extern "C" int nnis_chain(const void* layers, int layer_count, int m, int width, int heads, int kv_heads, int head_dim, int inner, int splits, int page_waves,
                          int gain_dtype, float eps, float scale, const float* x, float* x_out, void* y_out, const float* tok_cos, const float* tok_sin,
                          const int* tok_pos, const int* tok_page, const int* tok_pages, int max_pages, void* words, long long word_count, void* runs, long long run_count,
                          void* host_fail, void* stream_ptr) {
  NNIS_REQUIRE(head_dim == HD && fits(m, width, heads, kv_heads, inner, splits), "chain: %d rows, width %d, %d/%d heads of %d, inner %d, %d runs are not taken", m,
               width, heads, kv_heads, head_dim, inner, splits);
  NNIS_REQUIRE(layers && x && x_out && y_out && tok_cos && tok_sin && tok_pos && tok_page && tok_pages && max_pages > 0 && words && host_fail, "chain: an operand is missing");
  long long runs_needed;
  const long long needed = nnis_chain_words(layer_count, m, width, heads, kv_heads, inner, splits, &runs_needed);
  NNIS_REQUIRE(needed > 0 && word_count == needed && run_count >= runs_needed && (runs || runs_needed == 0), "chain: %lld and %lld words for %d layers", word_count,
               run_count, layer_count);
  NNIS_REQUIRE(nnis_dtype_ok(gain_dtype) && eps > 0.0f && scale > 0.0f, "chain: bad gain type, eps or scale");
  for (const void* p : {(const void*)x, (const void*)x_out, (const void*)y_out, (const void*)tok_cos, (const void*)tok_sin, (const void*)words, (const void*)runs})
    NNIS_REQUIRE((uintptr_t)p % 16 == 0, "chain: operands must be 16-byte aligned");
  ChainArgs a;
  a.layers = (const ChainLayer*)layers; a.layer_count = layer_count;
  a.rows = m; a.tiles = (m + kMostRows - 1) / kMostRows; a.m = min(m, kMostRows);
  a.width = width; a.heads = heads; a.kv_heads = kv_heads; a.inner = inner; a.splits = splits; a.gain_dtype = gain_dtype;
  a.eps = eps; a.inv_width = 1.0f / (float)width; a.scale_log2 = scale * 1.4426950408889634f;
  a.x = x; a.x_out = x_out; a.y_out = (bf16_t*)y_out; a.tok_cos = tok_cos; a.tok_sin = tok_sin; a.tok_pos = tok_pos; a.tok_page = tok_page; a.tok_pages = tok_pages;
  a.max_pages = max_pages; a.words = (unsigned*)words; a.run_words = (unsigned*)runs;
  a.layer_words = lay_out(a);
  a.words_bytes = a.layer_words * layer_count * 4;
  a.run_bytes = a.layer_runs * layer_count * 4;
  a.fail = a.words + (word_count - 32);
  a.host_fail = (unsigned*)host_fail;
  // wide models' units are large: 8 waves share them
  const int waves = width > 1024 ? 8 : 4;
  NNIS_REQUIRE(page_waves == 1 || page_waves == 2 || page_waves == 4 || (page_waves == 8 && waves == 8), "chain: %d waves for a run's pages", page_waves);
  a.page_waves = page_waves;
  // The ways that the layers' kernels cut K for so few rows (nnis_gemm_fused, nnis_gemm_residual), so that a step's numbers are the
  // same bits by either route; four waves take up to four parts (narrow rows' are no more), and down's eight two a wave.
  auto cut = [&](int k, int depth, int strips, int most) {
    int parts = 1;
    while (parts < most && (k + 63) / 64 > parts * depth && strips * parts * 2 <= 4096) parts *= 2;
    return parts;
  };
  a.parts_first = cut(width, 2, 0, 8);
  a.parts_qkv = cut(width, 4, 0, waves);
  a.parts_out = cut(heads * HD, 4, 0, waves);
  a.parts_gate = cut(width, 4, inner / 8, waves);
  const bool alike = heads / kv_heads <= 4;  // (larger groups' scores are other bits in any case)
  if (waves == 8 && (a.parts_gate < 4 || !alike)) a.parts_gate = 8;  // (not the layers' bits there)
  a.parts_down = cut(inner, 4, 0, 8);
  a.down_paired = waves == 8 && alike && width <= 2048 && inner >= 80 * 64;
  const int units = waves == 8 ? units_of<8>() : units_of<4>();
  a.n_qkv = (heads + 2 * kv_heads) * 2 / units;
  const int last = m - (a.tiles - 1) * kMostRows;
  auto att = [&](int rows) { return rows * kv_heads * ((heads / kv_heads + 3) / 4) * splits; };
  a.runs_in_out = splits > 1 && splits <= 8 && m == 1 && heads <= 4 * waves;  // (so many heads are one round of K)
  auto comb = [&](int rows) { return splits > 1 && !a.runs_in_out ? (rows * heads + 4 * waves - 1) / (4 * waves) : 0; };
  a.n_att = att(a.m);
  a.n_att_all = (a.tiles - 1) * a.n_att + att(last);
  a.n_comb = comb(a.m);
  a.n_comb_all = (a.tiles - 1) * a.n_comb + comb(last);
  a.n_strip = width / 16;
  a.n_out = width / 16 / (waves == 8 ? into_units_of<8, false>() : into_units_of<4, false>());
  a.n_down = width / 16 / (waves == 8 ? into_units_of<8, true>() : into_units_of<4, true>());
  a.n_gate = inner / 16 / units;
  const long long blocks = m + (long long)layer_count * (a.tiles * (a.n_qkv + a.n_out + a.n_gate + a.n_down) + a.n_att_all + a.n_comb_all);
  NNIS_REQUIRE(blocks < (1LL << 30), "chain: too many blocks");
  hipStream_t stream = (hipStream_t)stream_ptr;
  if (chain_clear(words, word_count - 32, runs, runs_needed, a.fail, stream)) return 1;
  // (up to four rows a lane ends one element instead of four: 32/4 heads, 22 layers, width 2048, 1 row at 500 tokens 496 -> 475 us and 4 rows
  // 495 -> 490; 32/32 heads, 24 layers, one row 757 -> 747 and behind 3,000 tokens, whose runs `out` adds up, 847 -> 832)
  if (waves == 8 && m <= 4) hipLaunchKernelGGL((chain_kernel<8, 4, false, true>), dim3((unsigned)blocks), dim3(512), 0, stream, a);
  else if (waves == 8) hipLaunchKernelGGL((chain_kernel<8, 16, false, true>), dim3((unsigned)blocks), dim3(512), 0, stream, a);
  else if (m <= 4) hipLaunchKernelGGL((chain_kernel<4, 4, false, false>), dim3((unsigned)blocks), dim3(256), 0, stream, a);
  else if (m <= 8) hipLaunchKernelGGL((chain_kernel<4, 8, false, true>), dim3((unsigned)blocks), dim3(256), 0, stream, a);
  else if (a.tiles == 1) hipLaunchKernelGGL((chain_kernel<4, 16, false, true>), dim3((unsigned)blocks), dim3(256), 0, stream, a);
  else hipLaunchKernelGGL((chain_kernel<4, 16, true, true>), dim3((unsigned)blocks), dim3(256), 0, stream, a);
  NNIS_LAUNCH_CHECK("chain");
  return 0;
}
