// 32-bit matrix products on the matrix cores: Y[M, N] = X[M, K] * W[N, K]^T for 32-bit weights in the
// checkpoint's order (K contiguous in both operands).  For few rows with v_mfma_f32_16x16x4_f32: lane l holds row l % 16 of
// either operand at k = l / 16, and D[4 * (l / 16) + e][l % 16] of the result, e = 0..3.  Which k a (lane group,
// instruction) stands for is free as long as both operands agree: lane group g loads 4 consecutive k, 16 bytes,
// and instruction j of four takes the group's j-th, so that 16 bytes a lane are 16 k of 16 rows.  For tiles with
// v_mfma_f32_16x16x32_bf16 on operands split into three bfloat16 numbers each, whose sum they are (below).
//
// Operands enter with all their 24 bits and sums are 32-bit.  (Tiles leave the three smallest of the nine products of a term's parts
// out: 2^-24 of the term at most, 2^-27.5 in the root mean square, what rounding it once would take; what the parts do not hold
// goes through the 32-bit instruction.)  A sum's terms come in
// another order than in the ordered kernel (gemm.hip), in several shorter chains (a wave's share of K, or runs of
// kFlushSteps steps), so its error against 64 bits is smaller than the one long chain's: 509 x 2048 x 5632 of
// normal values, root mean square error over that of the result 4.8e-7 (few rows) and 2.5e-7 (tiles; 3.0e-7 with the 32-bit
// instruction, whose chains round 8 times in 32 k instead of 6) against 1.3e-6, 8 x 960 x 576 1.6e-7 and 2.2e-7 against 4.3e-7.
//
// What a product does with its sums: stores them, adds them to the residual stream, or, with strips of weight rows that
// belong together taken in pairs, gates them (silu(gate) * up) or rotates queries and keys and writes the cache
// (Fused).  The kernel for few rows also takes the RMS norm before the product: it multiplies x * gain, sums the
// squares of its share of a row on the way, and scales the sums by 1 / sqrt(mean + eps) at the end.
//
//  * gemm_f32_few_kernel: few rows of X (a decode step, a short prompt), or too few tiles to fill the chip.  The
//    weight is streamed straight into operand registers; the waves of a block share K and meet in LDS.
//  * gemm_f32_tiled_kernel: tiles of 32 to 128 rows and 64 to 128 columns, K in steps of 32 through two stages in LDS.
// Which of them, and so which chains, goes by the sizes: a row's last bits depend on how many rows the product has, where
// the ordered kernel's do not.
#include "common.h"

#include <type_traits>

namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;

__device__ __forceinline__ f32x4 load4(const float* p) { return *(const f32x4*)p; }
__device__ __forceinline__ f32x4 load4(const bf16_t* p) {
  const bf16x4 v = *(const bf16x4*)p;
  return (f32x4){(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}

// 16 k of a tile of 16 weight rows x 16 rows of X
__device__ __forceinline__ f32x4 multiply16(f32x4 w, f32x4 x, f32x4 sum) {
#pragma unroll
  for (int j = 0; j < 4; ++j) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(w[j], x[j], sum, 0, 0, 0);
  return sum;
}

enum : int { F32_STORE = 0, F32_SILU = 1, F32_ROPE = 2, F32_RESIDUAL = 3 };

struct Fused {
  void* y;  // stored: [m, n]; residual: the stream [m, n], added to in place; gated: [m, n / 2]; rotated: the queries [m, heads * head_dim]
  int y_dtype;        // stored only; else 32-bit
  const float* gain;  // [k]: the norm's weight (few rows), or null
  float eps;
  // rotation and cache (epilogue.h has the same for 16-bit pages)
  const float* cos_table;  // [positions, head_dim / 2]
  const float* sin_table;
  const int* tok_slot;
  const int* tok_pos;
  float* k_pages;  // null: this run keeps no cache of its own
  float* v_pages;
  const int* block_table;
  int max_pages, heads, kv_heads, head_dim;
  const float* tok_cos;  // the step's tables, all three or none: each token's rows of the rotation tables, its position's page
  const float* tok_sin;
  const int* tok_page;
};

// The weight row at place r of strip s (of ROWS rows) of a pair: the gate's row and the up projection's, or a row of the
// lower half of a head and its partner in the upper half.  -1: beyond the last.
template <int EPI, int ROWS>
__device__ __forceinline__ int paired_row(const Fused& f, int unit, int s, int r, int n) {
  const int j = unit * ROWS + r;
  if constexpr (EPI == F32_SILU) return j < n / 2 ? s * (n / 2) + j : -1;
  const int half = f.head_dim / 2;
  return j < n / 2 ? j / half * f.head_dim + s * half + j % half : -1;
}

struct TokenPlace {
  int pos, page;  // page < 0: nothing to write (a padding row, no cache)
};
__device__ __forceinline__ TokenPlace place_of(const Fused& f, int token) {
  TokenPlace p;
  p.pos = f.tok_pos[token];
  if (!f.k_pages) p.page = -1;
  else if (f.tok_page) p.page = f.tok_page[token];
  else {
    const int slot = f.tok_slot[token];
    p.page = slot >= 0 ? f.block_table[(size_t)slot * f.max_pages + p.pos / kPageTokens] : -1;
  }
  return p;
}

// four consecutive columns of a row of Y, those below n
__device__ __forceinline__ void store_columns(void* y, int y_dtype, int row, int column, int n, f32x4 v) {
  const size_t at = (size_t)row * n + column;
  if (column + 4 <= n && n % 4 == 0) {
    if (y_dtype == NNIS_F32) {
      *(f32x4*)((float*)y + at) = v;
    } else {
      bf16x4 narrow;
#pragma unroll
      for (int e = 0; e < 4; ++e) narrow[e] = (__bf16)v[e];
      *(bf16x4*)((bf16_t*)y + at) = narrow;
    }
  } else {
    for (int e = 0; e < 4; ++e)
      if (column + e < n) store_from_f32(y, y_dtype, at + e, v[e]);
  }
}

// the stream's four columns that a product is added to (asked for ahead of the sums), and the sum
__device__ __forceinline__ f32x4 ask_columns(const float* x, int row, int column, int n) {
  const size_t at = (size_t)row * n + column;
  if (column + 4 <= n && n % 4 == 0) return *(const f32x4*)(x + at);
  f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
  for (int e = 0; e < 4; ++e)
    if (column + e < n) v[e] = x[at + e];
  return v;
}

// a pair's sums of one token: lo and hi hold places 4 g .. 4 g + 3 (`first`) of the strips; pair: the unit
template <int EPI, int ROWS>
__device__ __forceinline__ void finish_pair(const Fused& f, int token, TokenPlace place, int unit, int first, int n, f32x4 lo, f32x4 hi) {
  const int j = unit * ROWS + first;
  if constexpr (EPI == F32_SILU) {
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = lo[e] / (1.0f + expf(-lo[e])) * hi[e];
    store_columns(f.y, NNIS_F32, token, j, n / 2, v);
  } else {
    const int hd = f.head_dim, half = hd / 2, head = j / half, at = j % half;
    if (j >= n / 2) return;
    if (head < f.heads + f.kv_heads) {  // queries and keys turn
      const f32x4 c = *(const f32x4*)((f.tok_cos ? f.tok_cos + (size_t)token * half : f.cos_table + (size_t)place.pos * half) + at);
      const f32x4 sn = *(const f32x4*)((f.tok_sin ? f.tok_sin + (size_t)token * half : f.sin_table + (size_t)place.pos * half) + at);
      const f32x4 turned_lo = lo * c - hi * sn, turned_hi = hi * c + lo * sn;
      if (head < f.heads) {
        float* to = (float*)f.y + ((size_t)token * f.heads + head) * hd + at;
        *(f32x4*)to = turned_lo;
        *(f32x4*)(to + half) = turned_hi;
      } else if (place.page >= 0) {
        float* to = f.k_pages + ((size_t)place.page * f.kv_heads + head - f.heads) * nnis_k_page_elems(hd);
        *(f32x4*)(to + nnis_k_offset(place.pos % kPageTokens, at)) = turned_lo;  // 4 channels lie within a chunk of 8
        *(f32x4*)(to + nnis_k_offset(place.pos % kPageTokens, at + half)) = turned_hi;
      }
    } else if (place.page >= 0) {
      float* to = f.v_pages + ((size_t)place.page * f.kv_heads + head - f.heads - f.kv_heads) * nnis_v_page_elems(hd);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        to[nnis_v_offset(at + e, place.pos % kPageTokens)] = lo[e];
        to[nnis_v_offset(at + half + e, place.pos % kPageTokens)] = hi[e];
      }
    }
  }
}

// a lane's share of a row on its way through the norm
__device__ __forceinline__ void norm_share(f32x4& x, f32x4 gain, float& square) {
  square += (x[0] * x[0] + x[1] * x[1]) + (x[2] * x[2] + x[3] * x[3]);
  x *= gain;
}

// ---- few rows -----------------------------------------------------------------------------------------------------
// A block owns S strips of 16 weight rows and NT tiles of 16 rows of X; its W waves take chunks of 16 k in turn (wave
// w the chunks w, w + W, ..: together they read a row's consecutive memory), up to U of a wave's chunks in flight at
// once.  A wave's last chunks, however many, are one round: every round is a trip to memory.
// HALF (up to 8 rows of X): a strip has 8 weight rows; lanes r < 8 and r >= 8 of a load hold the same rows at k that
// are 16 apart, in both operands, so that of the product D[i][j] the quarters i, j < 8 and i, j >= 8 are the sums
// of two halves of a chunk of 32 k (the other two quarters mean nothing).  Twice as many blocks for a product
// whose strips are few, and no lane loads what another one has.
template <typename XT, int S, int NT, int W, int U, bool HALF, bool NORM, int EPI>
__global__ __launch_bounds__(64 * W) void gemm_f32_few_kernel(const XT* __restrict__ x, const float* __restrict__ w, Fused f, int m, int n, int k) {
  static_assert(!HALF || NT == 1, "half strips are for up to 8 rows");
  constexpr bool kPaired = EPI == F32_SILU || EPI == F32_ROPE;
  static_assert(!kPaired || S == 2, "a pair is two strips");
  constexpr int ROWS = HALF ? 8 : 16, CHUNK = HALF ? 32 : 16;
  __shared__ f32x4 parts[W][S * NT][kWave];
  __shared__ float squares[NORM ? W : 1][NORM ? NT * 16 : 1];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int r = lane % 16, g = lane / 16;
  const int unit = blockIdx.x, row0 = blockIdx.y * NT * 16;
  const int k_lane = HALF ? (r / 8) * 16 + g * 4 : g * 4;  // this lane's first k of a chunk

  // rows beyond the ends read a valid row and are not stored
  const float* w_row[S];
  const XT* x_row[NT];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    int row;
    if constexpr (kPaired) row = paired_row<EPI, ROWS>(f, unit, s, r % ROWS, n);
    else row = (unit * S + s) * ROWS + r % ROWS;
    w_row[s] = w + (size_t)(row >= 0 && row < n ? row : n - 1) * k + k_lane;
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int row = row0 + t * 16 + r % ROWS;
    x_row[t] = x + (size_t)(row < m ? row : m - 1) * k + k_lane;
  }
  f32x4 sum[S][NT];
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int t = 0; t < NT; ++t) sum[s][t] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};
  float square[NT];  // of this lane's share of its rows
#pragma unroll
  for (int t = 0; t < NT; ++t) square[t] = 0.0f;
  const float* gain = NORM ? f.gain + k_lane : nullptr;
  // what the end needs of the rows a wave finishes is asked for now
  TokenPlace place[EPI == F32_ROPE ? NT : 1];
  if constexpr (EPI == F32_ROPE) {
#pragma unroll
    for (int t = 0; t < NT; ++t) place[t] = place_of(f, row0 + t * 16 + r < m ? row0 + t * 16 + r : m - 1);
  }

  int c = wave;
  auto round = [&](auto count) {  // this wave's next `count` chunks, none of which reaches beyond K
    constexpr int N = decltype(count)::value;
    f32x4 wv[N][S], xv[N][NT], gv[N];
#pragma unroll
    for (int u = 0; u < N; ++u) {
#pragma unroll
      for (int s = 0; s < S; ++s) wv[u][s] = load4(w_row[s] + (c + u * W) * CHUNK);
#pragma unroll
      for (int t = 0; t < NT; ++t) xv[u][t] = load4(x_row[t] + (c + u * W) * CHUNK);
      if constexpr (NORM) gv[u] = load4(gain + (c + u * W) * CHUNK);
    }
    if constexpr (NORM) {
#pragma unroll
      for (int u = 0; u < N; ++u)
#pragma unroll
        for (int t = 0; t < NT; ++t) norm_share(xv[u][t], gv[u], square[t]);
    }
#pragma unroll
    for (int u = 0; u < N; ++u)
#pragma unroll
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int t = 0; t < NT; ++t) sum[s][t] = multiply16(wv[u][s], xv[u][t], sum[s][t]);
    c += N * W;
  };
  const int whole = k / CHUNK;
  int left = whole > wave ? (whole - wave + W - 1) / W : 0;
  constexpr int kLast = U + U / 2;  // the last round takes up to this many
  for (; left > kLast; left -= U) round(std::integral_constant<int, U>());
#define NNIS_LAST_ROUND(N) \
  if constexpr (N <= kLast) { \
    if (left == N) round(std::integral_constant<int, N <= kLast ? N : 1>()); \
  }
  NNIS_LAST_ROUND(1) NNIS_LAST_ROUND(2) NNIS_LAST_ROUND(3) NNIS_LAST_ROUND(4) NNIS_LAST_ROUND(5) NNIS_LAST_ROUND(6)
  NNIS_LAST_ROUND(7) NNIS_LAST_ROUND(8) NNIS_LAST_ROUND(9) NNIS_LAST_ROUND(10) NNIS_LAST_ROUND(11) NNIS_LAST_ROUND(12)
#undef NNIS_LAST_ROUND
  static_assert(kLast <= 12, "a last round for every count");
  if (whole * CHUNK < k && whole % W == wave) {
    // K's last, partial chunk: lanes beyond K read their row's first k and count as zeros
    const bool in = whole * CHUNK + k_lane < k;
    const int at = in ? whole * CHUNK : -k_lane;
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 wv[S], xv[NT];
#pragma unroll
    for (int s = 0; s < S; ++s) wv[s] = load4(w_row[s] + at);
#pragma unroll
    for (int t = 0; t < NT; ++t) xv[t] = load4(x_row[t] + at);
#pragma unroll
    for (int s = 0; s < S; ++s) wv[s] = in ? wv[s] : zero;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      xv[t] = in ? xv[t] : zero;
      if constexpr (NORM) norm_share(xv[t], load4(gain + at), square[t]);
    }
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int t = 0; t < NT; ++t) sum[s][t] = multiply16(wv[s], xv[t], sum[s][t]);
  }

#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int t = 0; t < NT; ++t) parts[wave][s * NT + t][lane] = sum[s][t];
  if constexpr (NORM) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      if constexpr (HALF) square[t] += __shfl_xor(square[t], 8, kWave);  // the other half of the chunks
      square[t] += __shfl_xor(square[t], 16, kWave);
      square[t] += __shfl_xor(square[t], 32, kWave);
      if (g == 0) squares[wave][t * 16 + r] = square[t];
    }
  }
  // a wave adds up the parts, in their order, of a (strip, tile), or of a pair of strips and a tile
  constexpr int kItems = kPaired ? NT : S * NT;
  f32x4 held[EPI == F32_RESIDUAL ? (kItems + W - 1) / W : 1];
  if constexpr (EPI == F32_RESIDUAL) {
#pragma unroll
    for (int i = 0; i < (kItems + W - 1) / W; ++i) {
      const int item = wave + i * W, row = row0 + (item % NT) * 16 + r;
      if (item < kItems && row < m && (!HALF || (g < 2 && r < 8)))
        held[i] = ask_columns((const float*)f.y, row, (unit * S + item / NT) * ROWS + g * 4, n);
    }
  }
  __syncthreads();
  if (HALF && (g >= 2 || r >= 8)) return;  // (no barrier below)
  auto added = [&](int slot) {
    f32x4 total = parts[0][slot][lane];
    if constexpr (HALF) total += parts[0][slot][lane + 40];  // rows and columns 8 on
#pragma unroll
    for (int p = 1; p < W; ++p) {
      total += parts[p][slot][lane];
      if constexpr (HALF) total += parts[p][slot][lane + 40];
    }
    return total;
  };
#pragma unroll
  for (int i = 0; i < (kItems + W - 1) / W; ++i) {
    const int item = wave + i * W, t = item % NT, row = row0 + t * 16 + r;
    if (item >= kItems || row >= m) continue;
    float scale = 1.0f;
    if constexpr (NORM) {
      float total = squares[0][t * 16 + r];
#pragma unroll
      for (int p = 1; p < W; ++p) total += squares[p][t * 16 + r];
      scale = 1.0f / sqrtf(total / (float)k + f.eps);
    }
    if constexpr (kPaired) {
      static_assert(NT <= W, "a wave finishes one tile");
      f32x4 lo = added(t), hi = added(NT + t);
      if constexpr (NORM) {
        lo *= scale;
        hi *= scale;
      }
      TokenPlace at = place[0];
      if constexpr (EPI == F32_ROPE) {
#pragma unroll
        for (int u = 1; u < NT; ++u) at = u == t ? place[u] : at;
      }
      finish_pair<EPI, ROWS>(f, row, at, unit, g * 4, n, lo, hi);
    } else {
      f32x4 total = added(item);
      if constexpr (NORM) total *= scale;
      if constexpr (EPI == F32_RESIDUAL) total += held[i];
      store_columns(f.y, EPI == F32_RESIDUAL ? (int)NNIS_F32 : f.y_dtype, row, (unit * S + item / NT) * ROWS + g * 4, n, total);
    }
  }
}

// ---- tiles --------------------------------------------------------------------------------------------------------
constexpr int kStepK = 32;      // k of a step: 128 bytes of a row
constexpr int kFlushSteps = 8;  // a chain of sums is this many steps long, then goes into the total

extern __shared__ __align__(16) char f32_lds[];  // two stages of BM rows of X in three parts

// A 32-bit number as the sum of three of 8 significant bits: x = hi + mid + lo, exactly, wherever the last of its bits is at least
// bfloat16's smallest number, 2^-133: from 2^-110 on, and for whoever ends early.  Both differences are exact, and what lo stands
// for has bits behind the first 16 of its word just where lo does not hold it whole: `left` collects these words, and is 0 in
// its lower half as long as every number was the sum of its parts.  AT_ONCE: into `left` right behind the conversions; the compiler by
// itself keeps the words to the end of a step, which takes up to 36 registers more.  A number that is none, or that rounds up to
// infinity, leaves parts that make its product one that is none.
template <int COUNT>
struct Split {
  typedef __attribute__((ext_vector_type(COUNT))) __bf16 part;
  part hi, mid, lo;
};
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
__device__ __forceinline__ f32x2 widen(bf16x2 v) {
  const unsigned both = __builtin_bit_cast(unsigned, v);
  return (f32x2){__uint_as_float(both << 16), __uint_as_float(both & 0xffff0000u)};
}
template <bool AT_ONCE>
__device__ __forceinline__ Split<4> split4(f32x4 v, unsigned& left) {
  Split<4> out;
#pragma unroll
  for (int e = 0; e < 4; e += 2) {  // (two at a time: one conversion for both)
    const f32x2 x = {v[e], v[e + 1]};
    const bf16x2 hi = __builtin_convertvector(x, bf16x2);
    const f32x2 rest = x - widen(hi);
    const bf16x2 mid = __builtin_convertvector(rest, bf16x2);
    const f32x2 last = rest - widen(mid);
    const bf16x2 lo = __builtin_convertvector(last, bf16x2);
    if constexpr (AT_ONCE) asm("v_or3_b32 %0, %0, %1, %2" : "+v"(left) : "v"(last[0]), "v"(last[1]));
    else left |= __float_as_uint(last[0]) | __float_as_uint(last[1]);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      out.hi[e + i] = hi[i];
      out.mid[e + i] = mid[i];
      out.lo[e + i] = lo[i];
    }
  }
  return out;
}

// TN tiles of one 16 rows of X in 32 bits throughout, operands straight from memory (row, weights[j]: this lane's row of each): for
// what a sum of parts may not stand for.  In runs of kFlushSteps steps of 32 k like the parts' sums, DEPTH steps' operands in flight.
template <int TN, int DEPTH>
__device__ __forceinline__ void multiply_in_32_bits(const float* row, const float* const (&weights)[TN], int k, f32x4 (&total)[TN]) {
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  const int first = threadIdx.x % kWave / 16 * 4, full = k / kStepK;  // this lane group's k of 16; steps without k beyond the last
  struct Operands {
    f32x4 a[2], b[2][TN];
  };
  auto multiply = [&](const Operands& v, f32x4 (&sum)[TN]) {
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int j = 0; j < TN; ++j) sum[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(v.b[half][j][q], v.a[half][q], sum[j], 0, 0, 0);
  };
  f32x4 sum[TN];
#pragma unroll
  for (int j = 0; j < TN; ++j) sum[j] = total[j] = zero;
  if (full > 0) {
    auto ask = [&](Operands& v, int step) {  // (beyond the last full one: that one, which is not multiplied again)
      const int at = (step < full ? step : full - 1) * kStepK + first;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        v.a[half] = load4(row + at + half * 16);
#pragma unroll
        for (int j = 0; j < TN; ++j) v.b[half][j] = load4(weights[j] + at + half * 16);
      }
    };
    Operands ring[DEPTH];
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) ask(ring[d], d);
    int run = 0;
    auto flush = [&] {
      if (++run < kFlushSteps) return;
      run = 0;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        total[j] += sum[j];
        sum[j] = zero;
      }
    };
    int step = 0;
#pragma unroll 1
    for (; step + DEPTH <= full; step += DEPTH)
#pragma unroll
      for (int d = 0; d < DEPTH; ++d) {
        multiply(ring[d], sum);
        ask(ring[d], step + d + DEPTH);
        flush();
      }
#pragma unroll
    for (int d = 0; d < DEPTH - 1; ++d)
      if (step + d < full) {
        multiply(ring[d], sum);
        flush();
      }
  }
  if (full * kStepK < k) {
    Operands last;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int at = full * kStepK + half * 16 + first;
      last.a[half] = at < k ? load4(row + at) : zero;
#pragma unroll
      for (int j = 0; j < TN; ++j) last.b[half][j] = at < k ? load4(weights[j] + at) : zero;
    }
    multiply(last, sum);
  }
#pragma unroll
  for (int j = 0; j < TN; ++j) total[j] += sum[j];
}

// Whether a sum of parts stands: not if it is no number or infinite, nor so small that parts of its terms may be missing, which are no
// numbers below 2^-149 (a zero stays).
__device__ __forceinline__ bool parts_hold(float v) {
  const unsigned magnitude = __float_as_uint(v) & 0x7fffffffu;
  return magnitude == 0u || (magnitude >= 0x12000000u && magnitude < 0x7f800000u);  // from 2^-91 on
}

// Bytes of LDS of a tile's two stages and of its rows' and columns' marks, and the waves of a SIMD that they leave room for (and the
// registers have to).
constexpr int tile_stages(int rows, int columns, int groups) { return 2 * groups * (rows + columns) * kStepK * 3 * (int)sizeof(__bf16); }
constexpr int tile_lds(int rows, int columns, int groups) { return tile_stages(rows, columns, groups) + (rows + columns) * (int)sizeof(unsigned); }
constexpr int tile_waves(int lds, int waves) { return 160 * 1024 / lds * waves / 4; }

// KG groups of WGM x WGN waves; a wave has BM / WGM rows and BN / WGN columns, a group every KG-th run of 32 k.  On the 16-bit
// matrix instruction a term x w of a sum is the six largest products of the operands' parts: x_hi w_hi,
// x_hi w_mid, x_mid w_hi, x_mid w_mid, x_hi w_lo and x_lo w_hi (of x_mid w_lo, x_lo w_mid and x_lo w_lo none is above 2^-25 of it), six times the work at sixteen times the 32-bit instruction's
// rate.  The block's threads split each number once, on its way into LDS, where a stage has three planes of 16 rows by 32 k; a
// lane's 8 k of a step are the 16 bytes at k = 4 g and those at 16 + 4 g, g = l / 16, in both operands, and are read as one
// operand.  What bounds the kernel is the sum of what a SIMD issues: a step of a wave tile of 64 x 32 is 48 matrix instructions
// of 16 cycles, about 75 vector instructions (11 for two numbers split) and 26 of LDS, 2,600 cycles for two waves of the 3,050
// measured; neither half the conversions, loads that hit nearer, operands read a step ahead nor two groups that take turns
// (products of one beside reads of the other) changed it by more than 5%.  Where a block has a compute unit to itself two groups
// share K, so that a SIMD has two waves: 509 x 2048 x 5632 in 64 x 64 114 -> 90 us (106 with the 32-bit instruction);
// with several blocks a unit one group is as fast and meets less.  2000 x 11264 x 2048 in 128 x 128: 501 us, 184 TFLOP/s (the
// 32-bit instruction's peak is 157, its kernel reached 128); 509 x 11264 x 2048 196 -> 150; 509 x 2560 x 2048 57 -> 41.  The
// marks of rows whose numbers are not the sum of their parts are 1 to 4% of these times (side by side, without and with: 90.9 and 94.0, 507 and 514,
// 151 and 151, 42.8 and 43.5).
template <int BM, int BN, int WGM, int WGN, int KG, int EPI>
__global__ __launch_bounds__(64 * WGM * WGN * KG, tile_waves(tile_lds(BM, BN, KG), WGM * WGN * KG)) void gemm_f32_tiled_kernel(
    const float* __restrict__ x, const float* __restrict__ w, Fused f, int m, int n, int k, int col_blocks) {
  constexpr bool kPaired = EPI == F32_SILU || EPI == F32_ROPE;
  constexpr int THREADS = 64 * WGM * WGN * KG, WM = BM / WGM, WN = BN / WGN;
  static_assert(!kPaired || WN % 32 == 0, "a wave has whole pairs of strips");
  constexpr int TM = WM / 16, TN = WN / 16;  // tiles of 16 x 16 a wave has, each way
  constexpr int ROW_CHUNKS = 8 * KG, BLOCK_K = kStepK * KG;  // a step of the block
  constexpr int LOAD_ROWS = THREADS / ROW_CHUNKS;  // rows that one load of every thread brings
  constexpr int A_LOADS = (BM + LOAD_ROWS - 1) / LOAD_ROWS, B_LOADS = (BN + LOAD_ROWS - 1) / LOAD_ROWS;
  constexpr int PLANE = 512, TILE = 3 * PLANE;  // 16 rows of a part and of all parts, in elements
  constexpr int GROUP = (BM + BN) / 16 * TILE, STAGE = KG * GROUP;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int k_group = wave / (WGM * WGN), wave_m = wave / WGN % WGM, wave_n = wave % WGN;
  const int r = lane % 16, g = lane / 16;
  // blocks go to the 8 dies in turn: a die's blocks are consecutive tiles, rows fastest, so that its L2 holds a few
  // column blocks of W and the rows of X
  int row_block, col_block;
  {
    const int total = gridDim.x, die = blockIdx.x % 8, nth = blockIdx.x / 8;
    const int each = total / 8, more = total % 8;
    const int tile = die * each + (die < more ? die : more) + nth;
    const int row_blocks = total / col_blocks;
    row_block = tile % row_blocks;
    col_block = tile / row_blocks;
  }
  const int row0 = row_block * BM, col0 = col_block * BN;
  // the weight row at place `place` of the block's BN (pairs: strips 2 u and 2 u + 1 of 16 are unit u's); -1 or from n on: none
  auto weight_row = [&](int place) {
    if constexpr (kPaired) return paired_row<EPI, 16>(f, col_block * (BN / 32) + place / 32, place / 16 % 2, place % 16, n);
    else return col0 + place;
  };

  // Rows beyond the end: a valid one, not stored.  Loads go by a base that is the same in every lane (the tile's first row; the
  // first of the 8 weight rows of a wave's load, which follow one another) and an offset in bytes, and give zeros from the base's
  // limit on, the operand's end at most: that is where the last step's chunks beyond K are asked for, and steps beyond the last (they
  // are not multiplied, and zeros are the sum of their parts).
  constexpr unsigned kNowhere = 0xfffffff0u;
  auto limit_of = [](size_t elements) { return elements * 4 < kNowhere ? (unsigned)(elements * 4) : kNowhere; };
  const int steps = (k + BLOCK_K - 1) / BLOCK_K, full = k / BLOCK_K;
  const auto a_base = __builtin_amdgcn_make_buffer_rsrc((void*)(x + (size_t)row0 * k), 0, limit_of((size_t)(m - row0) * k), 0x00027000);
  const int load_row = threadIdx.x / ROW_CHUNKS, chunk = threadIdx.x % ROW_CHUNKS, group = chunk % 4;
  // chunk c (of 8) is half c / 4 of the 8 k of lane group c % 4; 16 rows' chunks of a group lie together, row ^ 2 group, so that the
  // two rows that 16 lanes write, and the 8 rows that 8 lanes read, lie in different banks
  const int place_in_tile = chunk / 8 * GROUP + group * 128 + chunk / 4 % 2 * 4;
  auto place_of_row = [&](int row) { return row / 16 * TILE + place_in_tile + (row % 16 ^ group * 2) * 8; };
  unsigned a_from[A_LOADS], b_from[B_LOADS];
  __amdgpu_buffer_rsrc_t b_base[B_LOADS];
#pragma unroll
  for (int o = 0; o < A_LOADS; ++o) {
    const int row = row0 + o * LOAD_ROWS + load_row;
    a_from[o] = (unsigned)(((row < m ? row : m - 1) - row0) * k + chunk * 4) * 4u;
  }
#pragma unroll
  for (int o = 0; o < B_LOADS; ++o) {
    const int row = weight_row(o * LOAD_ROWS + load_row), first = __builtin_amdgcn_readfirstlane(row);
    const int start = first >= 0 && first < n ? first : 0;
    b_base[o] = __builtin_amdgcn_make_buffer_rsrc((void*)(w + (size_t)start * k), 0, limit_of((size_t)(n - start) * k), 0x00027000);
    b_from[o] = (unsigned)((row >= 0 && row < n ? row - start : 0) * k + chunk * 4) * 4u;
  }
  __bf16* stages = (__bf16*)f32_lds;
  // which rows of X, and behind them which weight rows, hold numbers that are not the sum of their parts
  unsigned* lossy = (unsigned*)(f32_lds + tile_stages(BM, BN, KG));
  for (int i = threadIdx.x; i < BM + BN; i += THREADS) lossy[i] = 0u;
  unsigned a_left[A_LOADS], b_left[B_LOADS];
#pragma unroll
  for (int o = 0; o < A_LOADS; ++o) a_left[o] = 0u;
#pragma unroll
  for (int o = 0; o < B_LOADS; ++o) b_left[o] = 0u;

  // (the step's place in the vector offset: the check against the limit takes no other into account for certain)
  const int steps_there = full + (full * BLOCK_K + chunk * 4 < k ? 1 : 0);  // (a last, short one counts where this thread's chunk is in it)
  auto load = [&](__amdgpu_buffer_rsrc_t base, unsigned from, int step) {
    const unsigned at = step < steps_there ? from + (unsigned)step * (BLOCK_K * 4) : kNowhere;
    return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(base, (int)at, 0, 0));
  };
  auto in_tile = [&](int o, int rows) { return rows % LOAD_ROWS == 0 || o * LOAD_ROWS + load_row < rows; };
  struct Raw {
    f32x4 a[A_LOADS], b[B_LOADS];
  };
  auto ask = [&](Raw& v, int step) {
#pragma unroll
    for (int o = 0; o < A_LOADS; ++o)
      if (in_tile(o, BM)) v.a[o] = load(a_base, a_from[o], step);
#pragma unroll
    for (int o = 0; o < B_LOADS; ++o)
      if (in_tile(o, BN)) v.b[o] = load(b_base[o], b_from[o], step);
  };
  auto put = [&](f32x4 v, __bf16* to, unsigned& left) {
    // (two groups: a step's numbers are not to be waited for, and split, together with the step's before it: 41 -> 37 us; one: 4% slower)
    if constexpr (KG > 1) asm volatile("" : "+v"(v));
    // (two groups have registers for it and are 3% faster without; one: 96 x 96 would keep some in scratch memory)
    const Split<4> parts = split4<KG == 1>(v, left);
    *(bf16x4*)to = parts.hi;
    *(bf16x4*)(to + PLANE) = parts.mid;
    *(bf16x4*)(to + 2 * PLANE) = parts.lo;
  };
  auto stage_step = [&](const Raw& v, int stage) {
    __bf16* to = stages + stage * STAGE;
#pragma unroll
    for (int o = 0; o < A_LOADS; ++o)
      if (in_tile(o, BM)) put(v.a[o], to + place_of_row(o * LOAD_ROWS + load_row), a_left[o]);
#pragma unroll
    for (int o = 0; o < B_LOADS; ++o)
      if (in_tile(o, BN)) put(v.b[o], to + BM / 16 * TILE + place_of_row(o * LOAD_ROWS + load_row), b_left[o]);
  };

  f32x4 sum[TM][TN], total[TM][TN];
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) sum[i][j] = total[i][j] = zero;
  auto product = [](bf16x8 b, bf16x8 a, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a, c, 0, 0, 0); };
  auto read_part = [&](Split<8>& v, const __bf16* tile) {
    const __bf16* at = tile + g * 128 + (r ^ g * 2) * 8;
    v.hi = *(const bf16x8*)at;
    v.mid = *(const bf16x8*)(at + PLANE);
    v.lo = *(const bf16x8*)(at + 2 * PLANE);
  };
  auto meet = [] {  // every wave's reads and writes of LDS so far are done
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  struct Operands {
    Split<8> rows[TM], weights[TN];
  };
  auto read_step = [&](Operands& v, int stage) {
    const __bf16* from = stages + stage * STAGE + k_group * GROUP;
#pragma unroll
    for (int j = 0; j < TN; ++j) read_part(v.weights[j], from + BM / 16 * TILE + (wave_n * TN + j) * TILE);
#pragma unroll
    for (int i = 0; i < TM; ++i) read_part(v.rows[i], from + (wave_m * TM + i) * TILE);
  };
  auto multiply = [&](const Operands& v) {
#pragma unroll
    for (int term = 0; term < 6; ++term)  // the small ones first
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const bf16x8 of_w = term == 1 ? v.weights[j].lo : (term == 2 || term == 4 ? v.weights[j].mid : v.weights[j].hi);
          const bf16x8 of_x = term == 0 ? v.rows[i].lo : (term == 2 || term == 3 ? v.rows[i].mid : v.rows[i].hi);
          sum[i][j] = product(of_w, of_x, sum[i][j]);
        }
  };

  // Step s lies in stage s % 2.  It is asked for three steps ahead, split and put there one ahead.  A stage is filled again
  // behind the barrier behind its last reads.
  Raw raw[2];
  ask(raw[0], 0);
  ask(raw[1], 1);
  stage_step(raw[0], 0);
  ask(raw[0], 2);
  meet();
  int run = 0;
  auto one_step = [&](int step, Raw& next, int stage) {
    Operands here;
    read_step(here, stage);
    multiply(here);
    stage_step(next, 1 - stage);
    ask(next, step + 3);
    if (++run == kFlushSteps) {
      run = 0;
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          total[i][j] += sum[i][j];
          sum[i][j] = zero;
        }
    }
    meet();
  };
  int step = 0;
  for (; step + 1 < steps; step += 2) {
    one_step(step, raw[1], 0);
    one_step(step + 1, raw[0], 1);
  }
  if (step < steps) one_step(step, raw[1], 0);
#pragma unroll
  for (int o = 0; o < A_LOADS; ++o)
    if (in_tile(o, BM) && (a_left[o] & 0xffffu)) lossy[o * LOAD_ROWS + load_row] = 1u;
#pragma unroll
  for (int o = 0; o < B_LOADS; ++o)
    if (in_tile(o, BN) && (b_left[o] & 0xffffu)) lossy[BM + o * LOAD_ROWS + load_row] = 1u;
  meet();
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) total[i][j] += sum[i][j];
  if constexpr (KG > 1) {  // the groups' sums meet in LDS (all reads of the stages are behind the barrier)
    f32x4* sums = (f32x4*)f32_lds + (size_t)(wave % (WGM * WGN)) * TM * TN * kWave + lane;
    if (k_group != 0)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) sums[(i * TN + j) * kWave] = total[i][j];
    meet();
    if (k_group != 0) return;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) total[i][j] += sums[(i * TN + j) * kWave];
  }

  // A wave that has sums which do not stand, or rows or columns of numbers that are not the sum of their parts, takes their 16 rows
  // again in 32 bits, and those sums from there: 509 x 11264 x 2048 with one row of X that is no number 212 us, with nothing
  // else 590, without 173.  (One lane's chain for each such sum, one after the other: 3,716 and 22,655.)
  static_assert(TN * 4 <= 32, "a bit for each of a lane's sums of a row");
  unsigned lossy_columns = 0u;
#pragma unroll
  for (int j = 0; j < TN; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) lossy_columns |= lossy[BM + wave_n * WN + j * 16 + g * 4 + e] << (j * 4 + e);
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    unsigned again = lossy[wave_m * WM + i * 16 + r] ? ~0u : lossy_columns;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) again |= (parts_hold(total[i][j][e]) ? 0u : 1u) << (j * 4 + e);
    const int row = row0 + wave_m * WM + i * 16 + r;
    if (row - r >= m || !__any(again)) continue;  // (rows beyond the end, here and below: a valid one, not stored)
    const float* weights[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int of = weight_row(wave_n * WN + j * 16 + r);
      weights[j] = w + (size_t)(of >= 0 && of < n ? of : 0) * k;
    }
    f32x4 sums[TN];
    multiply_in_32_bits<TN, 2>(x + (size_t)(row < m ? row : m - 1) * k, weights, k, sums);
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (again >> (j * 4 + e) & 1u) total[i][j][e] = sums[j][e];
  }

#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int row = row0 + wave_m * WM + i * 16 + r;
    if (row >= m) continue;
    if constexpr (kPaired) {
      TokenPlace place = {0, -1};
      if constexpr (EPI == F32_ROPE) place = place_of(f, row);
#pragma unroll
      for (int u = 0; u < TN / 2; ++u)
        finish_pair<EPI, 16>(f, row, place, (col0 + wave_n * WN) / 32 + u, g * 4, n, total[i][2 * u], total[i][2 * u + 1]);
    } else {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int column = col0 + wave_n * WN + j * 16 + g * 4;
        f32x4 v = total[i][j];
        if constexpr (EPI == F32_RESIDUAL) v += ask_columns((const float*)f.y, row, column, n);
        store_columns(f.y, EPI == F32_RESIDUAL ? (int)NNIS_F32 : f.y_dtype, row, column, n, v);
      }
    }
  }
}

template <int EPI, bool NORM, typename XT, int S, int NT, int W, int U, bool HALF = false>
void launch_few(const XT* x, const float* w, const Fused& f, int m, int n, int k, hipStream_t stream) {
  const int rows = (HALF ? 8 : 16) * S;
  const dim3 grid((n + rows - 1) / rows, (m + 16 * NT - 1) / (16 * NT));
  hipLaunchKernelGGL((gemm_f32_few_kernel<XT, S, NT, W, U, HALF, NORM, EPI>), grid, dim3(64 * W), 0, stream, x, w, f, m, n, k);
}

template <int EPI, int BM, int BN, int WGM, int WGN, int KG>
int launch_tiled(const float* x, const float* w, const Fused& f, int m, int n, int k, hipStream_t stream) {
  constexpr int lds = tile_lds(BM, BN, KG);
  static_assert(lds <= 160 * 1024 && tile_stages(BM, BN, KG) >= BM * BN * 4, "a compute unit has 160 KB; the groups' sums fit before the marks");
  auto kernel = gemm_f32_tiled_kernel<BM, BN, WGM, WGN, KG, EPI>;
  NNIS_REQUIRE(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess,
               "gemm_f32: %d bytes of LDS were refused", lds);
  const int col_blocks = (n + BN - 1) / BN;
  const long long blocks = (long long)col_blocks * ((m + BM - 1) / BM);
  NNIS_REQUIRE(blocks < (1LL << 31), "gemm_f32: %d rows exceed the grid limit", m);
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(64 * WGM * WGN * KG), lds, stream, x, w, f, m, n, k, col_blocks);
  return 0;
}

// Which kernel a product takes.  Up to 16 rows the weight's bytes and the trips to memory set the time, measured with 8
// rows over cold weights, microseconds (32-bit; the ordered kernel in brackets): half strips while whole ones leave half
// the compute units without a block, 2048 x 5632 14.0 against 21 (295), 576 x 1536 5.9 against 7.2 (84), but 2560 x 2048 10.1 against
// 8.7; blocks of 4 waves where the strips are many, 11264 x 2048 21.9 against 24.5 (220); two strips a block beyond, 49152 x
// 576 27.7 against 29.1, 32000 x 2048 59.1 against 61.5.  Pairs of strips, with the norm before them: half strips up to 8 rows
// (576 wide, gated 3072 rows 6.0 against 7.2, rotated 960 6.5 against 7.4; 2048 wide, gated 11264 24.2 against 28.1; a 30-layer decode step of 8 sequences, 576 wide,
// 1.51 -> 1.12 ms with the norms, gates, rotations and sums in the products), then two strips up to 8192 rows of weight (16
// rows of 6144 x 2048 19.3 against 20.6).  Beyond 16 rows a variant's time is close to a start and, for every
// round of its blocks on 256 compute units, a slope times K: the least of these is taken.  Measured:
// 64 x 2048 x 2048 13.4 us (two strips, one tile a block), 100 x 2048 x 2048 18.1 (2 x 2; 23.9 in tiles of 32 x 64), 100 x 11264 x 2048
// 47.5 (tiles of 64 x 96; 53.6 in 128 x 64), 509 x 2048 x 5632 94 (64 x 64; 109 in 32 x 64), 2000 x 11264 x 2048 519 (128 x 128; 572 in 64 x 128).
// Over 7 weights from 960 x 576 to 11264 x 2048 at 20 to 2,000 rows the form taken is 0.2% slower than the best on average.
struct Variant {
  int rows, columns;  // of a block
  float slope, start; // microseconds: slope * K for each round of blocks, and start
};
constexpr Variant kVariants[] = {
    {16, 16, 0.0050f, 2.0f}, {16, 32, 0.0064f, 2.0f}, {32, 32, 0.0083f, 2.0f}, {64, 32, 0.0135f, 2.0f},
    {32, 64, 0.0095f, 4.0f}, {64, 64, 0.0145f, 4.5f}, {64, 96, 0.0185f, 4.5f}, {96, 64, 0.0190f, 4.5f}, {96, 96, 0.0285f, 3.5f},
    {64, 128, 0.0224f, 12.5f}, {128, 64, 0.0235f, 6.0f}, {128, 96, 0.0315f, 4.8f}, {128, 128, 0.0353f, 5.9f}};
constexpr int kFewVariants = 4, kCountVariants = sizeof(kVariants) / sizeof(kVariants[0]);
enum : int { kHalfStrips = kCountVariants, kFourWaves, kTwoStrips, kHints };

bool fits_pairs(int variant) {  // whole pairs of strips to a wave
  return variant >= kFewVariants && variant < kCountVariants ? kVariants[variant].columns % 64 == 0 : variant != 0;
}

int pick_variant(bool f32, bool pairs, int m, int n, int k) {
  if (m <= 16) {
    if (pairs) return m <= 8 ? kHalfStrips : (n <= 8192 ? kTwoStrips : kFourWaves);
    if (m <= 8 && n <= 2048) return kHalfStrips;
    return n <= 8192 ? 0 : (n < 24000 ? kFourWaves : kTwoStrips);
  }
  int best = -1;
  float least = 0.0f;
  for (int v = 0; v < (f32 ? kCountVariants : kFewVariants); ++v) {  // (rows in 16 bits are widened on their way into registers)
    if (pairs && !fits_pairs(v)) continue;
    const Variant& it = kVariants[v];
    const long long blocks = (long long)((m + it.rows - 1) / it.rows) * ((n + it.columns - 1) / it.columns);
    const float time = (float)((blocks + 255) / 256) * it.slope * (float)k + it.start;
    if (best < 0 || time < least) {
      best = v;
      least = time;
    }
  }
  return best;
}

template <int EPI, bool NORM, typename XT>
int run_variant(int variant, const XT* x, const float* w, const Fused& f, int m, int n, int k, hipStream_t s) {
  constexpr bool kPaired = EPI == F32_SILU || EPI == F32_ROPE;
  constexpr int S = kPaired ? 2 : 1;
  // (strips, tiles, waves, chunks in flight); (rows, columns, waves along either, groups)
  switch (variant) {
    case kHalfStrips: launch_few<EPI, NORM, XT, S, 1, 8, 4, true>(x, w, f, m, n, k, s); return 0;
    case kFourWaves: launch_few<EPI, NORM, XT, S, 1, 4, 8>(x, w, f, m, n, k, s); return 0;
    case kTwoStrips:
    case 1: launch_few<EPI, NORM, XT, 2, 1, 8, 4>(x, w, f, m, n, k, s); return 0;
    case 0:
      if constexpr (!kPaired) {
        launch_few<EPI, NORM, XT, 1, 1, 8, 4>(x, w, f, m, n, k, s);
        return 0;
      }
      break;
  }
  if constexpr (!NORM) {
    if (variant == 2) {
      launch_few<EPI, NORM, XT, 2, 2, 8, 4>(x, w, f, m, n, k, s);
      return 0;
    }
    if (variant == 3) {
      launch_few<EPI, NORM, XT, 2, 4, 4, 2>(x, w, f, m, n, k, s);
      return 0;
    }
    if constexpr (std::is_same<XT, float>::value) {
      switch (variant) {
        case 4: return launch_tiled<EPI, 32, 64, 2, 2, 2>(x, w, f, m, n, k, s);
        case 5: return launch_tiled<EPI, 64, 64, 2, 2, 2>(x, w, f, m, n, k, s);
        case 7: return launch_tiled<EPI, 96, 64, 2, 2, 2>(x, w, f, m, n, k, s);
        case 9: return launch_tiled<EPI, 64, 128, 1, 4, 1>(x, w, f, m, n, k, s);
        case 10: return launch_tiled<EPI, 128, 64, 2, 2, 2>(x, w, f, m, n, k, s);
        case 12: return launch_tiled<EPI, 128, 128, 2, 4, 1>(x, w, f, m, n, k, s);
      }
      if constexpr (!kPaired) {
        switch (variant) {
          case 6: return launch_tiled<EPI, 64, 96, 2, 2, 2>(x, w, f, m, n, k, s);
          case 8: return launch_tiled<EPI, 96, 96, 3, 2, 1>(x, w, f, m, n, k, s);
          case 11: return launch_tiled<EPI, 128, 96, 4, 2, 1>(x, w, f, m, n, k, s);
        }
      }
    }
  }
  return nnis_fail("gemm_f32: the form %d does not take this product", variant);
}

}  // namespace

constexpr int NNIS_GEMM_F32_NORM_ROWS = 16;  // the most rows whose norm the product takes itself

// Y = X W^T in 32 bits; `epilogue` (32-bit rows): 0 stored, 1 gated (y [m, n / 2]), 2 rotated and written into the cache (y
// [m, heads * head_dim]), 3 added to y [m, n].  `gain` (32-bit rows, up to 16 of them, epilogues 0 to 2): X stands for
// its RMS norm with this weight.  `hint`: one of the forms, -1 for the one that the sizes choose.
extern "C" int nnis_gemm_f32_fused(const void* x, int x_dtype, const float* gain, float eps, const float* w, void* y, int y_dtype, int m, int n,
                                   int k, int epilogue, const float* cos_table, const float* sin_table, const int* tok_slot, const int* tok_pos,
                                   float* k_pages, float* v_pages, const int* block_table, int max_pages, int heads, int kv_heads, int head_dim,
                                   const float* tok_cos, const float* tok_sin, const int* tok_page, int hint, void* stream) {
  NNIS_REQUIRE(nnis_dtype_ok(x_dtype) && nnis_dtype_ok(y_dtype), "gemm_f32: unknown dtype (x %d, y %d)", x_dtype, y_dtype);
  NNIS_REQUIRE(m >= 0 && n > 0 && k > 0 && k % 4 == 0, "gemm_f32: bad sizes m=%d n=%d k=%d (K a multiple of 4)", m, n, k);
  NNIS_REQUIRE(((uintptr_t)x | (uintptr_t)w | (uintptr_t)y | (uintptr_t)gain) % 16 == 0, "gemm_f32: operands must be 16-byte aligned");
  const bool f32 = x_dtype == NNIS_F32, pairs = epilogue == F32_SILU || epilogue == F32_ROPE;
  NNIS_REQUIRE(epilogue >= F32_STORE && epilogue <= F32_RESIDUAL && (epilogue == F32_STORE || (f32 && y_dtype == NNIS_F32)),
               "gemm_f32: no epilogue %d for these types", epilogue);
  NNIS_REQUIRE(gain == nullptr || (f32 && m <= NNIS_GEMM_F32_NORM_ROWS && epilogue != F32_RESIDUAL), "gemm_f32: the norm of %d rows is not taken", m);
  NNIS_REQUIRE(epilogue != F32_SILU || n % 2 == 0, "gemm_f32: %d rows are no gate and up projection", n);
  if (epilogue == F32_ROPE) {
    NNIS_REQUIRE(heads > 0 && kv_heads > 0 && head_dim > 0 && head_dim % 32 == 0 && n == (heads + 2 * kv_heads) * head_dim,
                 "gemm_f32: %d rows are not %d + 2 x %d heads of %d channels (a multiple of 32)", n, heads, kv_heads, head_dim);
    NNIS_REQUIRE(tok_pos && tok_slot && cos_table && sin_table && (k_pages == nullptr) == (v_pages == nullptr) && (!k_pages || (block_table && max_pages > 0)),
                 "gemm_f32: the rotation's operands are incomplete");
    NNIS_REQUIRE((tok_cos == nullptr) == (tok_sin == nullptr) && (tok_cos == nullptr) == (tok_page == nullptr), "gemm_f32: the step's tables come together");
    NNIS_REQUIRE(((uintptr_t)cos_table | (uintptr_t)sin_table | (uintptr_t)tok_cos | (uintptr_t)tok_sin | (uintptr_t)k_pages | (uintptr_t)v_pages) % 16 == 0,
                 "gemm_f32: the rotation's operands must be 16-byte aligned");
  }
  NNIS_REQUIRE(hint >= -1 && hint < kHints && (hint != kHalfStrips || m <= 8) && (hint < 0 || !pairs || fits_pairs(hint)),
               "gemm_f32: no variant %d for %d rows", hint, m);
  const int variant = hint >= 0 ? hint : pick_variant(f32, pairs, m, n, k);
  NNIS_REQUIRE(f32 || variant < kFewVariants || variant >= kCountVariants, "gemm_f32: tiles take 32-bit rows");
  NNIS_REQUIRE(variant >= kFewVariants || (m + kVariants[variant].rows - 1) / kVariants[variant].rows <= 65535, "gemm_f32: %d rows exceed the grid limit", m);
  if (m == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const Fused f = {y, y_dtype, gain, eps, cos_table, sin_table, tok_slot, tok_pos, k_pages, v_pages, block_table, max_pages,
                   heads, kv_heads, head_dim, tok_cos, tok_sin, tok_page};
  const float* x32 = (const float*)x;
  int status;
  if (!f32) status = run_variant<F32_STORE, false>(variant, (const bf16_t*)x, w, f, m, n, k, s);
  else if (epilogue == F32_RESIDUAL) status = run_variant<F32_RESIDUAL, false>(variant, x32, w, f, m, n, k, s);
  else if (epilogue == F32_SILU) status = gain ? run_variant<F32_SILU, true>(variant, x32, w, f, m, n, k, s) : run_variant<F32_SILU, false>(variant, x32, w, f, m, n, k, s);
  else if (epilogue == F32_ROPE) status = gain ? run_variant<F32_ROPE, true>(variant, x32, w, f, m, n, k, s) : run_variant<F32_ROPE, false>(variant, x32, w, f, m, n, k, s);
  else status = gain ? run_variant<F32_STORE, true>(variant, x32, w, f, m, n, k, s) : run_variant<F32_STORE, false>(variant, x32, w, f, m, n, k, s);
  if (status) return status;
  NNIS_LAUNCH_CHECK("gemm_f32");
  return 0;
}

extern "C" int nnis_gemm_f32(const void* x, int x_dtype, const float* w, void* y, int y_dtype, int m, int n, int k, int hint, void* stream) {
  return nnis_gemm_f32_fused(x, x_dtype, nullptr, 0.0f, w, y, y_dtype, m, n, k, F32_STORE, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, 0,
                             0, 0, nullptr, nullptr, nullptr, hint, stream);
}
