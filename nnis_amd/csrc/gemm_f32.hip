// 32-bit matrix products on the matrix cores: Y[M, N] = X[M, K] * W[N, K]^T for 32-bit weights in the
// checkpoint's order (K contiguous in both operands), with v_mfma_f32_16x16x4_f32: lane l holds row l % 16 of
// either operand at k = l / 16, and D[4 * (l / 16) + e][l % 16] of the result, e = 0..3.  Which k a (lane group,
// instruction) stands for is free as long as both operands agree: lane group g loads 4 consecutive k, 16 bytes,
// and instruction j of four takes the group's j-th, so that 16 bytes a lane are 16 k of 16 rows.
//
// The instruction multiplies and adds in 32 bits; nothing is rounded to fewer on the way.  A sum's terms come in
// another order than in the ordered kernel (gemm.hip), in several shorter chains (a wave's share of K, or runs of
// kFlushSteps steps), so its error against 64 bits is smaller than the one long chain's: 509 x 2048 x 5632 of
// normal values, root mean square error over that of the result 4.8e-7 (few rows) and 3.0e-7 (tiles) against 1.3e-6,
// 8 x 960 x 576 1.6e-7 and 2.8e-7 against 4.3e-7.
//
// What a product does with its sums: stores them, adds them to the residual stream, or, with strips of weight rows that
// belong together taken in pairs, gates them (silu(gate) * up) or rotates queries and keys and writes the cache
// (Fused).  The kernel for few rows also takes the RMS norm before the product: it multiplies x * gain, sums the
// squares of its share of a row on the way, and scales the sums by 1 / sqrt(mean + eps) at the end.
//
//  * gemm_f32_few_kernel: few rows of X (a decode step, a short prompt), or too few tiles to fill the chip.  The
//    weight is streamed straight into operand registers; the waves of a block share K and meet in LDS.
//  * gemm_f32_tiled_kernel: tiles of 32 to 128 rows and 64 to 128 columns, K in steps of 32 through a ring of stages in LDS.
// Which of them, and so which chains, goes by the sizes: a row's last bits depend on how many rows the product has, where
// the ordered kernel's do not.
#include "common.h"
#include "lds_loads.h"

#include <type_traits>

namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;

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
constexpr int kStepK = 32;      // k of a step: 128 bytes of a row, 8 chunks of 16 bytes
constexpr int kFlushSteps = 8;  // a chain of sums is this many steps long, then goes into the total

extern __shared__ __align__(16) char f32_lds[];  // NS stages of BM rows of X and BN rows of W

// 4 waves, 2 x 2, each with BM / 2 rows and BN / 2 columns.  A load instruction of a wave brings 8 rows of 128 bytes
// straight into LDS, lane l's 16 bytes to row l / 8, place l % 8; place p of row r holds chunk p ^ (r % 8), so that
// the 16 rows which a lane group reads together lie in different banks.  The matrix instructions bound the kernel (a
// step of a wave tile of 32 x 32 is 32 of them, 1,024 cycles, for 8 KB read from LDS and a quarter of 16 KB loaded).
template <int BM, int BN, int NS, int EPI>
__global__ __launch_bounds__(256) void gemm_f32_tiled_kernel(const float* __restrict__ x, const float* __restrict__ w, Fused f, int m, int n,
                                                             int k, int col_blocks) {
  constexpr bool kPaired = EPI == F32_SILU || EPI == F32_ROPE;
  static_assert(!kPaired || BN % 64 == 0, "a wave has whole pairs of strips");
  constexpr int TM = BM / 32, TN = BN / 32;  // tiles of 16 x 16 a wave has, each way
  constexpr int A_LOADS = BM / 32, B_LOADS = BN / 32, LOADS = A_LOADS + B_LOADS;  // load instructions a wave and step
  constexpr int A_BYTES = BM * kStepK * 4, STAGE_BYTES = (BM + BN) * kStepK * 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int wave_m = wave / 2, wave_n = wave % 2;
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

  const int chunk_k = ((lane % 8) ^ (lane / 8)) * 4;  // the first k of this lane's chunk of a step
  // rows in bytes from the tile's first row, and from the first of the wave's weight rows (of its pairs' lower or upper rows:
  // a wave's loads take the one or all the other), which are the same in every lane
  const float* a_base = x + (size_t)row0 * k;
  const float* b_base = w;
  int a_off[A_LOADS], b_off[B_LOADS], base_row = 0;
#pragma unroll
  for (int o = 0; o < A_LOADS; ++o) {
    const int row = (o * 4 + wave) * 8 + lane / 8;
    a_off[o] = (row0 + row < m ? row : m - 1 - row0) * k * 4;
  }
#pragma unroll
  for (int o = 0; o < B_LOADS; ++o) {
    const int in_tile = (o * 4 + wave) * 8 + lane / 8;  // (pairs: strips 2 u and 2 u + 1 of the tile are unit u's)
    int row;
    if constexpr (kPaired) row = paired_row<EPI, 16>(f, col_block * (BN / 32) + in_tile / 32, in_tile / 16 % 2, in_tile % 16, n);
    else row = col0 + in_tile;
    if (o == 0) {
      const int first = __builtin_amdgcn_readfirstlane(row);
      base_row = first >= 0 && first < n ? first : n - 1;
      b_base = w + (size_t)base_row * k;
    }
    b_off[o] = (row >= 0 && row < n ? row - base_row : 0) * k * 4;  // (rows beyond the end: a valid one, not stored)
  }
  // Step s lies in stage s % NS.  A step beyond the end, and the last step's chunks beyond K, are asked for from the
  // row's first chunk: valid memory; the former nobody reads, the latter count as zeros.
  const int steps = (k + kStepK - 1) / kStepK;
  auto ask = [&](int step, int stage) {
    char* base = f32_lds + stage * STAGE_BYTES + wave * 1024;
    const int at = step * kStepK + chunk_k;
    const int from = (at < k ? at : 0) * 4;
#pragma unroll
    for (int o = 0; o < A_LOADS; ++o) load_to_lds(a_base, a_off[o] + from, 0, base + o * 4096);
#pragma unroll
    for (int o = 0; o < B_LOADS; ++o) load_to_lds(b_base, b_off[o] + from, 0, base + A_BYTES + o * 4096);
  };

  f32x4 sum[TM][TN], total[TM][TN];
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) sum[i][j] = total[i][j] = zero;

  auto read_half = [&](int from, int half, f32x4 (&a)[TM], f32x4 (&b)[TN]) {
    const f32x4* a_tile = (const f32x4*)(f32_lds + from * STAGE_BYTES);
    const f32x4* b_tile = (const f32x4*)(f32_lds + from * STAGE_BYTES + A_BYTES);
    const int place = (half * 4 + g) ^ (r % 8);
#pragma unroll
    for (int i = 0; i < TM; ++i) a[i] = a_tile[(wave_m * (BM / 2) + i * 16 + r) * 8 + place];
#pragma unroll
    for (int j = 0; j < TN; ++j) b[j] = b_tile[(wave_n * (BN / 2) + j * 16 + r) * 8 + place];
  };
  auto multiply = [&](const f32x4 (&a)[TM], const f32x4 (&b)[TN]) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) sum[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(b[j][q], a[i][q], sum[i][j], 0, 0, 0);
  };

#pragma unroll
  for (int s = 0; s < NS - 1; ++s) ask(s, s);
  wait_loads_but<(NS - 2) * LOADS>();
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  int stage = 0;
  f32x4 a0[TM], b0[TN], a1[TM], b1[TN];
  // A step asks for the step NS - 1 ahead into the stage that was read a step ago, reads its second half under the
  // first half's products, and multiplies the second half behind the barrier, while the next step's first half is read.
  // Every read of a stage is waited for before the barrier that lets the stage be filled again.
  read_half(0, 0, a0, b0);
  const int full = k % kStepK == 0 ? steps : steps - 1;  // steps without chunks beyond K
  int run = 0;
  for (int step = 0; step < full; ++step) {
    ask(step + NS - 1, stage == 0 ? NS - 1 : stage - 1);
    read_half(stage, 1, a1, b1);
    multiply(a0, b0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    wait_loads_but<(NS - 2) * LOADS>();
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    stage = stage + 1 == NS ? 0 : stage + 1;
    read_half(stage, 0, a0, b0);  // (behind the last step: of a stage that nobody multiplies)
    multiply(a1, b1);
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
  }
  if (full < steps) {  // the last step: its chunks beyond K count as zeros
    const int k0 = full * kStepK + g * 4;
    read_half(stage, 1, a1, b1);
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      a0[i] = k0 < k ? a0[i] : zero;
      a1[i] = k0 + 16 < k ? a1[i] : zero;
    }
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      b0[j] = k0 < k ? b0[j] : zero;
      b1[j] = k0 + 16 < k ? b1[j] : zero;
    }
    multiply(a0, b0);
    multiply(a1, b1);
  }
  wait_loads_but<0>();  // the steps asked for beyond the end: nothing of this block is in flight when it ends

#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int row = row0 + wave_m * (BM / 2) + i * 16 + r;
    if (row >= m) continue;
    if constexpr (kPaired) {
      TokenPlace place = {0, -1};
      if constexpr (EPI == F32_ROPE) place = place_of(f, row);
#pragma unroll
      for (int u = 0; u < TN / 2; ++u)
        finish_pair<EPI, 16>(f, row, place, col_block * (BN / 32) + wave_n * (TN / 2) + u, g * 4, n, total[i][2 * u] + sum[i][2 * u],
                             total[i][2 * u + 1] + sum[i][2 * u + 1]);
    } else {
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int column = col0 + wave_n * (BN / 2) + j * 16 + g * 4;
        f32x4 v = total[i][j] + sum[i][j];
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

template <int EPI, int BM, int BN, int NS>
int launch_tiled(const float* x, const float* w, const Fused& f, int m, int n, int k, hipStream_t stream) {
  constexpr int lds = NS * (BM + BN) * kStepK * 4;
  static_assert(lds <= 160 * 1024, "a compute unit has 160 KB");
  auto kernel = gemm_f32_tiled_kernel<BM, BN, NS, EPI>;
  NNIS_REQUIRE(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess,
               "gemm_f32: %d bytes of LDS were refused", lds);
  const int col_blocks = (n + BN - 1) / BN;
  const long long blocks = (long long)col_blocks * ((m + BM - 1) / BM);
  NNIS_REQUIRE(blocks < (1LL << 31), "gemm_f32: %d rows exceed the grid limit", m);
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), lds, stream, x, w, f, m, n, k, col_blocks);
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
// 64 x 2048 x 2048 14.0 us (two strips, one tile a block), 128 x 2048 x 2048 18.7 (2 x 2), 128 x 11264 x 2048 60 (tiles of 64 x 96; 75
// in 64 x 64), 509 x 2048 x 5632 112 (64 x 64), 4000 x 11264 x 2048 1,443 (128 x 128; 128 TFLOP/s of the instruction's 157).
struct Variant {
  int rows, columns;  // of a block
  float slope, start; // microseconds: slope * K for each round of blocks, and start
};
constexpr Variant kVariants[] = {
    {16, 16, 0.0050f, 2.0f}, {16, 32, 0.0064f, 2.0f}, {32, 32, 0.0083f, 2.0f}, {64, 32, 0.0135f, 2.0f},
    {32, 64, 0.0105f, 3.5f}, {64, 64, 0.0189f, 3.5f}, {64, 96, 0.0280f, 3.5f}, {96, 64, 0.0280f, 3.5f}, {96, 96, 0.0405f, 3.5f},
    {64, 128, 0.0365f, 3.5f}, {128, 64, 0.0365f, 3.5f}, {128, 96, 0.0540f, 3.5f}, {128, 128, 0.0700f, 3.5f}};
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
  // (strips, tiles, waves, chunks in flight); (rows, columns, stages)
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
        case 4: return launch_tiled<EPI, 32, 64, 3>(x, w, f, m, n, k, s);
        case 5: return launch_tiled<EPI, 64, 64, 3>(x, w, f, m, n, k, s);
        case 7: return launch_tiled<EPI, 96, 64, 3>(x, w, f, m, n, k, s);
        case 9: return launch_tiled<EPI, 64, 128, 3>(x, w, f, m, n, k, s);
        case 10: return launch_tiled<EPI, 128, 64, 3>(x, w, f, m, n, k, s);
        case 12: return launch_tiled<EPI, 128, 128, 2>(x, w, f, m, n, k, s);
      }
      if constexpr (!kPaired) {
        switch (variant) {
          case 6: return launch_tiled<EPI, 64, 96, 3>(x, w, f, m, n, k, s);
          case 8: return launch_tiled<EPI, 96, 96, 3>(x, w, f, m, n, k, s);
          case 11: return launch_tiled<EPI, 128, 96, 3>(x, w, f, m, n, k, s);
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
