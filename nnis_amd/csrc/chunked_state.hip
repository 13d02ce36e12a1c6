// Recurrences over a matrix state, 64 tokens at a time on the 32-bit matrix instructions: the gated delta rule and
// retention over prompts (recurrent.hip has the same a token at a time, for single tokens and other sizes).
//
// Per head, S [key channels, value channels], a chunk of tokens t = 1 .. 64 from the state S0, c_t the product of the
// decays g_1 .. g_t (kept as a sum of logarithms: only quotients c_t / c_s of s <= t are taken, which are at most one):
//   S_t = c_t S0 + sum_{s <= t} (c_t / c_s) k_s u_s^T
//   o_t = c_t S0^T q_t + sum_{s <= t} (c_t / c_s) (k_s . q_t) u_s
// Retention has u = v.  The delta rule's u_t = beta_t (v_t - g_t S_(t-1)^T k_t) is, with the first line put in,
//   u_t + sum_{s < t} A_ts u_s = beta_t v_t - beta_t c_t S0^T k_t,   A_ts = beta_t (c_t / c_s) (k_t . k_s)
// so that with T = (I + A)^-1 (unit lower triangular)
//   U = V' - K' S0,   V' = T (beta v),   K' = T (beta c k).
// T, V' and K' need no state: a first kernel makes them for all chunks side by side, with M_ts = (c_t / c_s) (k_s . q_t)
// and the keys transposed and scaled by c_64 / c_s.  The second kernel walks the chunks of a (sequence, head, 16 value columns):
//   U = V' - K' S,   O = c (Q S) + M U,   S <- c_64 S + K~ U
// All of it is 32-bit (v_mfma_f32_16x16x4_f32 multiplies and adds in 32 bits).  A lane (r = l % 16, g = l / 16) holds
// rows 4 g + e of column r of a result; as the second operand of instruction e of the next product that is row 4 g + e
// of a sum over rows, if the first operand's lane group g brings its column 4 g + e: results go on as operands where
// they lie, and a first operand is 16 consecutive bytes a lane.
//
// Why: the recurrence a token at a time is a chain of 0.39 us a token and sequence for the delta rule, whatever the chip
// has free; a chunk of 64 is one of 4 us, beside 30 us for the first kernel and the ends.  Microseconds, a prompt of 300 /
// 1,500 tokens: the delta rule on 16 heads of 128 x 128 57 / 135 (130 / 602 a token at a time), retention on 8 heads of
// 128 x 256 25 / 74 (78 / 187, in pieces); 8 prompts of 2,048: 1,020 (1,500) and 421 (1,480).  What bounds the walk is the
// chain of a chunk: two products that wait for each other over U, two barriers, and a state that goes round through LDS.
// Error of the outputs against 64 bits, 1e-7 of their root mean square, and of a token at a time: delta rule, 16 heads of 128 x
// 128, decays of which most are forgotten within a few tokens 1.17 (1.17), slow ones 1.63 (2.52), between 1.38 (1.36); 4 heads of 16
// x 48 between 1.31 (1.25); retention 1.95 (5.11) over 1,500 tokens, 1.11 (1.15) over 20.  The states' are within 1% of a token
// at a time's, 1% above at fast decays, and half as large at slow ones.  (With a token's own M_tt u_t among the products, a twentieth
// of the time less, fast decays 1.20, between 1.41, 20 tokens of retention 1.20.)
#include "common.h"

namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;

constexpr int kChunk = 64;       // tokens of a chunk: four tiles of 16, one a wave
constexpr int kTiles = kChunk / 16;
constexpr int kGates = 2 * kChunk + 16;  // floats a (chunk, head) has for c_t, M_tt and c_64

__device__ __forceinline__ f32x4 mfma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// 16 rows of a sum: first operand `a` (four of its columns a lane), second the result tile `b`
__device__ __forceinline__ f32x4 multiply16(f32x4 a, f32x4 b, f32x4 sum) {
#pragma unroll
  for (int e = 0; e < 4; ++e) sum = mfma(a[e], b[e], sum);
  return sum;
}

__device__ __forceinline__ f32x4 sum8(const f32x4 (&p)[8]) { return ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7])); }

// Products with a tile on the diagonal, whose first operand is zero above it: a token that is infinite or no number must not
// reach the tokens before it (zero times it would be no number), so a tile that holds one is added up element by element.
// `a` as a first operand, `b` and the sum as results; what `a` holds on and above its diagonal is zero.
__device__ __forceinline__ f32x4 multiply_below(f32x4 a, f32x4 b, int lane) {
  const f32x4 none = b * 0.0f;
  f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
  if (__builtin_expect(!__any(!((none[0] + none[1]) + (none[2] + none[3]) == 0.0f)), 1)) {
    // (four chains: a row's nearest tokens, the largest terms, come last in one of them and not in the middle of a long one)
    const f32x4 p0 = mfma(a[0], b[0], sum), p1 = mfma(a[1], b[1], sum), p2 = mfma(a[2], b[2], sum), p3 = mfma(a[3], b[3], sum);
    return (p0 + p1) + (p2 + p3);
  }
  const int r = lane % 16, g = lane / 16;
#pragma unroll
  for (int e = 0; e < 4; ++e)
#pragma unroll 1
    for (int from = 0; from < 4; ++from) {  // column 4 from + e of a, row 4 from + e of b
      const float right = __shfl(b[e], from * 16 + r, kWave);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 4 * g + i, column = 4 * from + e;
        const float left = __shfl(a[e], from * 16 + row, kWave);
        sum[i] = column < row ? fmaf(left, right, sum[i]) : sum[i];
      }
    }
  return sum;
}

__device__ __forceinline__ f32x4 load4(const float* p) { return *(const f32x4*)p; }
__device__ __forceinline__ f32x4 load4(const bf16_t* p) {
  const bf16x4 v = *(const bf16x4*)p;
  return (f32x4){(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
}

struct ChunkArgs {
  const int* seq_slot;
  const int* seq_start;
  int batch, heads, key_dim, value_dim;
  // What the first kernel leaves, by (chunk, head); chunks are counted through the step's sequences.  Matrices lie as the
  // second kernel's waves load them: tiles of 16 x 16 as first operands, `operand_at`, 1 KB of consecutive memory a load.
  // (In rows, the step's stride of 4 and 8 KB between tokens put a load's 16 rows on one channel of the L2: 3.2 and 5 us a
  // chunk for retention and the delta rule.)
  float* within;   // [4 tiles of rows][4 of columns]: M below its diagonal
  float* keys_t;   // [key_dim / 16][4 tiles of tokens]: K~
  float* gates;    // [kGates]: c_t, then M_tt, then c_64
  float* queries;  // [4 tiles of tokens][key_dim / 16]
  float* keys;     // [4][key_dim / 16]: -K'  (delta rule)
  float* values;   // [value_dim / 16][4]: V' (delta rule), tiles as results
  // retention's values as the projection left them
  const void* v;
  int v_stride;
  float* state;
  size_t state_row, state_column;  // of an element of a head's state
  float* out;  // [tokens, heads * value_dim]
};

// where element (row, column) of a tile lies as a first operand: lane 16 (column / 4) + row, place column % 4
__device__ __forceinline__ int operand_at(int row, int column) { return ((column / 4) * 16 + row) * 4 + column % 4; }
constexpr int kTileFloats = 256;

// the sequence and the chunk of it that the step's chunk `c` is; false beyond the last
__device__ __forceinline__ bool find_chunk(const int* seq_start, int batch, int c, int& first, int& count) {
  for (int b = 0; b < batch; ++b) {
    const int n = seq_start[b + 1] - seq_start[b], chunks = (n + kChunk - 1) / kChunk;
    if (c < chunks) {
      first = seq_start[b] + c * kChunk;
      count = min(kChunk, n - c * kChunk);
      return true;
    }
    c -= chunks;
  }
  return false;
}

// ---- the second kernel ----------------------------------------------------------------------------------------------
// A block of eight waves has a sequence's head and 16 value columns.  Every wave holds the whole state of those columns (KT
// tiles of 16 key channels) and brings one tile of it up to date; waves 0 to 3 make U, a tile of the chunk's tokens each,
// waves 4 to 7 the outputs.  U and the new state go round through LDS.  A chunk's operands are asked for while the chunk before
// is worked on, in registers of their own: with both halves of the work in one wave they were 280 of them, and the
// compiler put the loads off until they were needed.
constexpr int kScanWaves = 8;

template <int KT, bool DELTA, typename V, bool OUTPUTS>
__device__ __forceinline__ void walk_chunks(const ChunkArgs& a, int head, int column, int begin, int end, int chunk0, int wave, int lane, float* state,
                                            f32x4 (*u_shared)[kWave], f32x4 (*s_shared)[kWave]) {
  static_assert(KT <= kScanWaves, "a wave has one tile of the state");
  constexpr bool kRows = OUTPUTS || DELTA;  // rows of a first operand that meets the state: queries, or -K'
  const int g = lane / 16, tile = wave % kTiles, e = a.value_dim;
  const int own = min(wave, KT - 1);  // the tile of the state that this wave brings up to date (wave < KT)
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  f32x4 S[KT], mine;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
#pragma unroll
    for (int t = 0; t < KT; ++t) S[t][i] = state[(size_t)(t * 16 + g * 4 + i) * a.state_row];
    mine[i] = state[(size_t)(own * 16 + g * 4 + i) * a.state_row];
  }

  struct Operands {
    f32x4 rows[kRows ? KT : 1], kt[kTiles], m[OUTPUTS ? kTiles : 1], own, v;  // v: the values, or c_t of the outputs' rows; own: their M_tt
    float c_end;
  };
  // (no load behind a branch: it would be waited for at once)
  auto load = [&](Operands& o, int chunk) {
    const size_t at = (size_t)(chunk0 + chunk) * a.heads + head;
    if constexpr (kRows) {
      const float* from = (OUTPUTS ? a.queries : a.keys) + ((at * kTiles + tile) * KT * kWave + lane) * 4;
#pragma unroll
      for (int t = 0; t < KT; ++t) o.rows[t] = load4(from + t * kTileFloats);
    }
    const float* kt = a.keys_t + ((at * KT + own) * kTiles * kWave + lane) * 4;
#pragma unroll
    for (int s = 0; s < kTiles; ++s) o.kt[s] = load4(kt + s * kTileFloats);
    if constexpr (OUTPUTS) {
      const float* m = a.within + ((at * kTiles + tile) * kTiles * kWave + lane) * 4;
#pragma unroll
      for (int s = 0; s < kTiles; ++s) o.m[s] = load4(m + (s == kTiles - 1 ? tile : min(s, tile)) * kTileFloats);  // (the last: on the diagonal)
      o.v = load4(a.gates + at * kGates + tile * 16 + g * 4);
      o.own = load4(a.gates + at * kGates + kChunk + tile * 16 + g * 4);
    } else if constexpr (DELTA) {
      o.v = load4(a.values + (((at * (e / 16) + column / 16) * kTiles + tile) * kWave + lane) * 4);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // (tokens beyond the end: a value that is there, zeroed where it is used)
        const int token = min(begin + chunk * kChunk + tile * 16 + g * 4 + i, end - 1);
        o.v[i] = to_f32(((const V*)a.v)[(size_t)token * a.v_stride + (size_t)head * e + column]);
      }
    }
    o.c_end = *(const __attribute__((address_space(4))) float*)(uintptr_t)(a.gates + at * kGates + 2 * kChunk);  // (a scalar load)
  };
  auto step = [&](const Operands& o, int chunk) {
    f32x4 sum = zero;
    if constexpr (kRows) {
      // eight short chains, added up afterwards: a third of the rounding of one long one, and no product waits for another
      f32x4 part[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) part[i] = zero;
#pragma unroll
      for (int t = 0; t < KT; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i) part[t % 2 * 4 + i] = mfma(o.rows[t][i], S[t][i], part[t % 2 * 4 + i]);
      sum = sum8(part);
    }
    if constexpr (!OUTPUTS && DELTA) u_shared[tile][lane] = o.v + sum;
    if constexpr (!OUTPUTS && !DELTA) {
      f32x4 v;
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = begin + chunk * kChunk + tile * 16 + g * 4 + i < end ? o.v[i] : 0.0f;
      u_shared[tile][lane] = v;
    }
    __syncthreads();
    f32x4 U[kTiles];
#pragma unroll
    for (int s = 0; s < kTiles; ++s) U[s] = u_shared[s][lane];
    const f32x4 u = u_shared[tile][lane];  // (of the outputs' own tokens)
    f32x4 part[kTiles];
#pragma unroll
    for (int s = 0; s < kTiles; ++s) part[s] = multiply16(o.kt[s], U[s], zero);
    mine = mine * o.c_end + ((part[0] + part[1]) + (part[2] + part[3]));
    if (wave < KT) s_shared[wave][lane] = mine;
    if constexpr (OUTPUTS) {
      // a token's own update comes last and once: where states are forgotten within a few tokens it is most of the output
      f32x4 within = zero;
#pragma unroll
      for (int s = 0; s < kTiles - 1; ++s)
        if (s < tile) within += multiply16(o.m[s], U[s], zero);
      within += multiply_below(o.m[kTiles - 1], u, lane);
      const f32x4 out = o.own * u + (sum * o.v + within);
      const int token = begin + chunk * kChunk + tile * 16 + g * 4;
      float* to = a.out + ((size_t)token * a.heads + head) * e + column;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (token + i < end) to[(size_t)i * a.heads * e] = out[i];
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < KT; ++t) S[t] = s_shared[t][lane];
  };
  const int chunks = (end - begin + kChunk - 1) / kChunk;
  Operands one, other;
  load(one, 0);
  for (int chunk = 0; chunk < chunks; chunk += 2) {
    load(other, min(chunk + 1, chunks - 1));
    __builtin_amdgcn_sched_barrier(0);  // (left to itself the compiler asks for them when they are needed)
    step(one, chunk);
    if (chunk + 1 >= chunks) break;
    load(one, min(chunk + 2, chunks - 1));
    __builtin_amdgcn_sched_barrier(0);
    step(other, chunk + 1);
  }
  if (wave < KT) {
#pragma unroll
    for (int i = 0; i < 4; ++i) state[(size_t)(wave * 16 + g * 4 + i) * a.state_row] = mine[i];
  }
}

template <int KT, bool DELTA, typename V>
__global__ __launch_bounds__(kWave * kScanWaves) void chunk_scan_kernel(ChunkArgs a) {
  __shared__ f32x4 u_shared[kTiles][kWave];
  __shared__ f32x4 s_shared[KT][kWave];
  // (heads vary fastest: blocks go to the 8 dies in turn, so that, of a multiple of 8 heads, the blocks of one run on one
  // die, whose L2 then holds what they all read)
  const int b = blockIdx.z, head = blockIdx.x;
  const int slot = a.seq_slot[b];
  if (slot < 0) return;
  const int begin = a.seq_start[b], end = a.seq_start[b + 1];
  if (end <= begin) return;
  int chunk0 = 0;
  for (int i = 0; i < b; ++i) chunk0 += (a.seq_start[i + 1] - a.seq_start[i] + kChunk - 1) / kChunk;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int column = blockIdx.y * 16 + lane % 16;
  float* state = a.state + ((size_t)slot * a.heads + head) * KT * 16 * a.value_dim + (size_t)column * a.state_column;
  if (wave < kTiles) walk_chunks<KT, DELTA, V, false>(a, head, column, begin, end, chunk0, wave, lane, state, u_shared, s_shared);
  else walk_chunks<KT, DELTA, V, true>(a, head, column, begin, end, chunk0, wave, lane, state, u_shared, s_shared);
}

// ---- the first kernel, delta rule -----------------------------------------------------------------------------------
struct DeltaChunkArgs {
  ChunkArgs c;
  const float* unit;  // [tokens, groups, 2, key_dim]: q (scaled) then k, unit vectors
  const float* dots;  // [tokens, groups]: q . k
  const void* rows;   // v of token t, head h at rows + t * stride + v_at + h * value_dim
  int dtype, stride, v_at, groups;
  const float* ba;  // [tokens, 2 * heads]
  const float* rate;
  const float* dt_bias;
};

// A block of eight waves has a (chunk, head): the gates by a lane a token; the ten tiles of K K^T and Q K^T on and below
// the diagonal; the inverses of the four tiles on A's diagonal, a wave each, by substitution; then the columns of [beta c k | beta v], 16 at a time, down
// the four row tiles: X_i = T_ii (R_i - sum_{j < i} A_ij X_j).
constexpr int kPrepareWaves = 8;

template <int KT>
__global__ __launch_bounds__(kWave * kPrepareWaves) void chunk_delta_prepare_kernel(DeltaChunkArgs a) {
  constexpr int d = KT * 16, kRow = kChunk + 4;
  __shared__ double logs[kChunk];  // sums in 64 bits: a quotient of two late tokens must not feel a great decay before them
  __shared__ float betas[kChunk];
  __shared__ __align__(16) float A[kChunk][kRow];     // -A, below the diagonal
  __shared__ __align__(16) float T[kTiles][16][20];   // the diagonal tiles' inverses, without their diagonal of ones
  constexpr int kUnitRow = d + 4;
  extern __shared__ __align__(16) float lds[];        // [2][64][kUnitRow]: queries, keys; zeros beyond the chunk's end
  int first, count;
  if (!find_chunk(a.c.seq_start, a.c.batch, blockIdx.x, first, count)) return;
  const int head = blockIdx.y, heads = a.c.heads, e = a.c.value_dim;
  const size_t at = (size_t)blockIdx.x * heads + head;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int r = lane % 16, g = lane / 16;
  const int qk_head = head / (heads / a.groups);
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};

  for (int i = threadIdx.x; i < kChunk * 2 * (d / 4); i += kWave * kPrepareWaves) {  // (a token's two rows lie together)
    const int token = i / (2 * (d / 4)), c = i % (2 * (d / 4));
    const f32x4 v = token < count ? load4(a.unit + ((size_t)(first + token) * a.groups + qk_head) * 2 * d + c * 4) : zero;
    *(f32x4*)(lds + (c < d / 4 ? 0 : kChunk * kUnitRow) + token * kUnitRow + c % (d / 4) * 4) = v;
  }
  if (wave == 0) {
    float log_g = 0.0f, beta = 0.0f;  // (tokens beyond the chunk's end change nothing)
    if (lane < count) {
      const float* ba = a.ba + (size_t)(first + lane) * 2 * heads;
      const float z = ba[heads + head] + a.dt_bias[head];
      log_g = -a.rate[head] * (z > 20.0f ? z : log1pf(expf(z)));
      // (a decay to zero: differences of infinite logarithms would be no numbers, and the decays behind a very large one would
      // drown in the sum; expf gives zero from -104 on)
      log_g = log_g < -1000.0f ? -1000.0f : log_g;
      beta = 1.0f / (1.0f + expf(-ba[head]));
    }
    double total = (double)log_g;
#pragma unroll
    for (int offset = 1; offset < kWave; offset *= 2) {
      const double before = __shfl_up(total, offset, kWave);
      total += lane >= offset ? before : 0.0;
    }
    logs[lane] = total;
    betas[lane] = beta;
    a.c.gates[at * kGates + lane] = expf((float)total);
    // (the one that a token at a time takes: summed with less rounding than M's products)
    a.c.gates[at * kGates + kChunk + lane] = lane < count ? a.dots[(size_t)(first + lane) * a.groups + qk_head] : 0.0f;
    if (lane == kChunk - 1) a.c.gates[at * kGates + 2 * kChunk] = expf((float)total);
  }
  __syncthreads();

  auto unit_row = [&](int token, int which) { return lds + which * kChunk * kUnitRow + token * kUnitRow; };
  for (int pair = wave; pair < kTiles * (kTiles + 1) / 2; pair += kPrepareWaves) {
    const int row_tile = pair < 1 ? 0 : (pair < 3 ? 1 : (pair < 6 ? 2 : 3)), s = pair - row_tile * (row_tile + 1) / 2;
    const float* k = unit_row(row_tile * 16 + r, 1) + g * 4;
    const float* q = unit_row(row_tile * 16 + r, 0) + g * 4;
    const float* other = unit_row(s * 16 + r, 1) + g * 4;
    f32x4 kk = zero, qk = zero, kk_part[8], qk_part[8];
#pragma unroll
    for (int t = 0; t < KT; ++t) {
      if (t % 4 == 0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) kk_part[i] = qk_part[i] = zero;
      }
      const f32x4 right = load4(other + t * 16), left_k = load4(k + t * 16), left_q = load4(q + t * 16);
      if (s == row_tile) *(f32x4*)(a.c.queries + (((at * kTiles + row_tile) * KT + t) * kWave + lane) * 4) = left_q;  // as it is an operand
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        kk_part[t % 2 * 4 + i] = mfma(left_k[i], right[i], kk_part[t % 2 * 4 + i]);
        qk_part[t % 2 * 4 + i] = mfma(left_q[i], right[i], qk_part[t % 2 * 4 + i]);
      }
      if (t % 4 == 3 || t == KT - 1) {
        kk += sum8(kk_part);
        qk += sum8(qk_part);
      }
    }
    {
      const int column = s * 16 + r;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int token = row_tile * 16 + g * 4 + i;
        const bool live = token < count && column < count;
        const bool met = live && column < token;
        const float ratio = met ? expf((float)(logs[token] - logs[column])) : 0.0f;
        A[token][column] = met ? -betas[token] * ratio * kk[i] : 0.0f;
        a.c.within[((at * kTiles + row_tile) * kTiles + s) * kTileFloats + operand_at(g * 4 + i, r)] = met ? ratio * qk[i] : 0.0f;
      }
    }
  }
  __syncthreads();

  if (wave < kTiles) {  // column r of the inverse of I + A's tile (wave, wave): x_i = [i = r] - sum_{s < i} A_is x_s
    float x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float v = i == r ? 1.0f : 0.0f;
#pragma unroll
      for (int s = 0; s < i; ++s) v = fmaf(A[wave * 16 + i][wave * 16 + s], x[s], v);
      x[i] = v;
    }
    if (g == 0)
#pragma unroll
      for (int i = 0; i < 16; ++i) T[wave][i][r] = i == r ? 0.0f : x[i];
  }
  __syncthreads();

  f32x4 t_rows[kTiles], a_rows[kTiles][kTiles];
#pragma unroll
  for (int i = 0; i < kTiles; ++i) {
    t_rows[i] = *(const f32x4*)&T[i][r][g * 4];
#pragma unroll
    for (int j = 0; j < i; ++j) a_rows[i][j] = *(const f32x4*)&A[i * 16 + r][j * 16 + g * 4];
  }
  f32x4 key_factor[kTiles], value_factor[kTiles];
#pragma unroll
  for (int i = 0; i < kTiles; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int token = i * 16 + g * 4 + j;
      value_factor[i][j] = betas[token];
      key_factor[i][j] = -betas[token] * expf((float)logs[token]);
    }
  for (int tile = wave; tile < KT + e / 16; tile += kPrepareWaves) {
    const bool is_key = tile < KT;
    const int column = (is_key ? tile : tile - KT) * 16 + r;
    f32x4 right[kTiles], x[kTiles];
#pragma unroll
    for (int i = 0; i < kTiles; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int token = i * 16 + g * 4 + j;  // (beyond the end: zeros)
        const float v = is_key ? unit_row(token, 1)[column]
                               : load_as_f32(a.rows, a.dtype, (size_t)(first + min(token, count - 1)) * a.stride + a.v_at + (size_t)head * e + column);
        right[i][j] = token < count ? v : 0.0f;
      }
#pragma unroll
    for (int i = 0; i < kTiles; ++i) {
      // (small terms first, the large one last: half the rounding of sums that start from it)
      f32x4 above = zero;
#pragma unroll
      for (int j = 0; j < i; ++j) above += multiply16(a_rows[i][j], x[j], zero);
      above += right[i] * (is_key ? key_factor[i] : value_factor[i]);
      x[i] = above + multiply_below(t_rows[i], above, lane);
      if (is_key) {
        float* to = a.c.keys + ((at * kTiles + i) * KT + tile) * kTileFloats;
#pragma unroll
        for (int j = 0; j < 4; ++j) to[operand_at(g * 4 + j, r)] = x[i][j];
      } else {
        *(f32x4*)(a.c.values + (((at * (e / 16) + tile - KT) * kTiles + i) * kWave + lane) * 4) = x[i];
      }
    }
  }
  // the keys transposed, a lane a token, times c_64 / c_s
  const float rest = expf((float)(logs[kChunk - 1] - logs[lane]));
  const float* key = unit_row(lane, 1);
  for (int c = wave * 4; c < d; c += 4 * kPrepareWaves) {
    const f32x4 v = load4(key + c);
    float* to = a.c.keys_t + ((at * KT + c / 16) * kTiles + lane / 16) * kTileFloats;
#pragma unroll
    for (int i = 0; i < 4; ++i) to[operand_at(c % 16 + i, lane % 16)] = v[i] * rest;
  }
}

// ---- the first kernel, retention --------------------------------------------------------------------------------------
struct RetentionChunkArgs {
  ChunkArgs c;
  const void* q;  // row t, head h: q + t * q_stride + h * key_dim
  const void* k;
  int q_stride, k_stride;
  float scale;
  const float* head_decay;  // [2, heads]: the decays, then their logarithms
  const float* rot_cos;     // the first rot_dim channels turn by the token's position, channel i with i + rot_dim / 2
  const float* rot_sin;
  const int* tok_pos;
  int rot_dim, rot_positions;
};

// A block has a (chunk, head): queries and keys widened, turned and scaled on their way into LDS; the queries written out;
// M, a wave a tile of rows; the keys transposed and scaled.  Decays are powers of one number, taken as exp(n log a).
template <int KT, typename T>
__global__ __launch_bounds__(256) void chunk_retention_prepare_kernel(RetentionChunkArgs a) {
  constexpr int d = KT * 16, kRow = d + 4;
  extern __shared__ __align__(16) float lds[];  // [2][64][kRow]: queries, keys
  int first, count;
  if (!find_chunk(a.c.seq_start, a.c.batch, blockIdx.x, first, count)) return;
  const int head = blockIdx.y, heads = a.c.heads;
  const size_t at = (size_t)blockIdx.x * heads + head;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
  const int r = lane % 16, g = lane / 16;
  const float log_of = a.head_decay[heads + head], log_a = log_of < -1e30f ? -1e30f : log_of;  // (a decay of zero: 0 times its logarithm)
  const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
  float* qs = lds;
  float* ks = lds + kChunk * kRow;

  const int half = a.rot_dim / 2;
  for (int i = threadIdx.x; i < kChunk * (d / 4); i += 256) {  // four channels of a token
    const int token = i / (d / 4), c = i % (d / 4) * 4;
    f32x4 q = zero, k = zero;
    if (token < count) {
      const T* q_row = (const T*)a.q + (size_t)(first + token) * a.q_stride + (size_t)head * d;
      const T* k_row = (const T*)a.k + (size_t)(first + token) * a.k_stride + (size_t)head * d;
      q = load4(q_row + c);
      k = load4(k_row + c);
      if (c < a.rot_dim) {
        const bool low = c < half;
        const int pair = low ? c : c - half, partner = low ? c + half : c - half;
        int pos = a.tok_pos[first + token];
        pos = pos < 0 ? 0 : (pos < a.rot_positions ? pos : a.rot_positions - 1);
        const f32x4 cos = load4(a.rot_cos + (size_t)pos * half + pair);
        f32x4 sin = load4(a.rot_sin + (size_t)pos * half + pair);
        if (low) sin = -sin;
        q = q * cos + load4(q_row + partner) * sin;
        k = k * cos + load4(k_row + partner) * sin;
      }
      q *= a.scale;
    }
    *(f32x4*)(a.c.queries + (((at * kTiles + token / 16) * KT + c / 16) * kWave + c % 16 / 4 * 16 + token % 16) * 4) = q;
    *(f32x4*)(qs + token * kRow + c) = q;
    *(f32x4*)(ks + token * kRow + c) = k;
  }
  if (wave == 0) {
    a.c.gates[at * kGates + lane] = expf((float)(lane + 1) * log_a);
    if (lane == 0) a.c.gates[at * kGates + 2 * kChunk] = expf((float)count * log_a);
  }
  __syncthreads();
  {
    const float* q_row = qs + (wave * 16 + r) * kRow + g * 4;
    f32x4 q[KT];
#pragma unroll
    for (int t = 0; t < KT; ++t) q[t] = load4(q_row + t * 16);
#pragma unroll
    for (int s = 0; s < kTiles; ++s) {
      if (s > wave) break;
      const float* k_row = ks + (s * 16 + r) * kRow + g * 4;
      f32x4 qk = zero, part[8];
#pragma unroll
      for (int t = 0; t < KT; ++t) {
        if (t % 4 == 0) {
#pragma unroll
          for (int i = 0; i < 8; ++i) part[i] = zero;
        }
        const f32x4 right = load4(k_row + t * 16);
#pragma unroll
        for (int i = 0; i < 4; ++i) part[t % 2 * 4 + i] = mfma(q[t][i], right[i], part[t % 2 * 4 + i]);
        if (t % 4 == 3 || t == KT - 1) qk += sum8(part);
      }
      const int column = s * 16 + r;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int token = wave * 16 + g * 4 + i;
        a.c.within[((at * kTiles + wave) * kTiles + s) * kTileFloats + operand_at(g * 4 + i, r)] =
            column < token ? expf((float)(token - column) * log_a) * qk[i] : 0.0f;
        if (column == token) a.c.gates[at * kGates + kChunk + token] = qk[i];
      }
    }
  }
  const float rest = lane < count ? expf((float)(count - 1 - lane) * log_a) : 0.0f;
  for (int c = wave * 4; c < d; c += 16) {
    const f32x4 v = load4(ks + lane * kRow + c);
    float* to = a.c.keys_t + ((at * KT + c / 16) * kTiles + lane / 16) * kTileFloats;
#pragma unroll
    for (int i = 0; i < 4; ++i) to[operand_at(c % 16 + i, lane % 16)] = v[i] * rest;
  }
}

size_t floats_a_chunk(int key_dim, int value_dim, bool delta) {
  return (size_t)kChunk * kChunk + 2 * (size_t)key_dim * kChunk + kGates + (delta ? (size_t)kChunk * (key_dim + value_dim) : 0);
}

void lay_out(ChunkArgs& c, float* scratch, int chunks, bool delta) {
  const size_t items = (size_t)chunks * c.heads;
  c.within = scratch;
  c.keys_t = c.within + items * kChunk * kChunk;
  c.gates = c.keys_t + items * kChunk * c.key_dim;
  c.queries = c.gates + items * kGates;
  c.keys = delta ? c.queries + items * kChunk * c.key_dim : nullptr;
  c.values = delta ? c.keys + items * kChunk * c.key_dim : nullptr;
}

}  // namespace

extern "C" int nnis_chunked_takes(int key_dim, int value_dim) {
  return key_dim > 0 && key_dim % 16 == 0 && key_dim <= 128 && value_dim > 0 && value_dim % 16 == 0;
}

// floats of scratch for a step of `tokens` rows in `batch` sequences (at most tokens / 64 + batch chunks)
extern "C" long long nnis_chunked_scratch(int tokens, int batch, int heads, int key_dim, int value_dim, int delta) {
  const long long chunks = tokens / kChunk + batch;
  return chunks * heads * (long long)floats_a_chunk(key_dim, value_dim, delta != 0);
}

#define NNIS_KEY_TILES(RUN)  \
  switch (key_dim / 16) {    \
    case 1: RUN(1); break;   \
    case 2: RUN(2); break;   \
    case 3: RUN(3); break;   \
    case 4: RUN(4); break;   \
    case 5: RUN(5); break;   \
    case 6: RUN(6); break;   \
    case 7: RUN(7); break;   \
    default: RUN(8); break;  \
  }

// The gated delta rule over a step's prompts, behind delta_prepare_kernel (nnis_gated_delta has the operands).
int nnis_gated_delta_chunks(const float* unit, const float* dots, const void* rows, int dtype, int stride, const float* ba, const float* rate, const float* dt_bias,
                            float* state, const int* seq_slot, const int* seq_start, int batch, int tokens, int heads, int groups, int key_dim,
                            int value_dim, float* out, float* scratch, hipStream_t s) {
  NNIS_REQUIRE(nnis_chunked_takes(key_dim, value_dim), "gated_delta: heads of %d and %d channels are not taken in chunks", key_dim, value_dim);
  const int chunks = tokens / kChunk + batch;
  DeltaChunkArgs a;
  ChunkArgs& c = a.c;
  c.seq_slot = seq_slot; c.seq_start = seq_start; c.batch = batch; c.heads = heads; c.key_dim = key_dim; c.value_dim = value_dim;
  lay_out(c, scratch, chunks, true);
  c.v = nullptr; c.v_stride = 0;
  c.state = state; c.state_row = 1; c.state_column = key_dim; c.out = out;
  a.unit = unit; a.dots = dots; a.rows = rows; a.dtype = dtype; a.stride = stride; a.v_at = 2 * groups * key_dim; a.groups = groups;
  a.ba = ba; a.rate = rate; a.dt_bias = dt_bias;
  const size_t lds = 2 * kChunk * (size_t)(key_dim + 4) * sizeof(float);
#define NNIS_RUN(KT)                                                                                                                       \
  NNIS_REQUIRE(hipFuncSetAttribute((const void*)chunk_delta_prepare_kernel<KT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)      \
                   == hipSuccess, "gated_delta: %zu bytes of LDS were refused", lds);                                                      \
  hipLaunchKernelGGL(chunk_delta_prepare_kernel<KT>, dim3(chunks, heads), dim3(kWave * kPrepareWaves), lds, s, a);                         \
  hipLaunchKernelGGL((chunk_scan_kernel<KT, true, float>), dim3(heads, value_dim / 16, batch), dim3(kWave * kScanWaves), 0, s, c)
  NNIS_KEY_TILES(NNIS_RUN)
#undef NNIS_RUN
  NNIS_LAUNCH_CHECK("gated_delta (chunks)");
  return 0;
}

// Retention over a step's prompts: nnis_gla_scan_turned with head_decay, in chunks.  Rows and tables in whole quarters of
// 16 (8 for bfloat16 rows) bytes: q, k and their strides and rot_dim / 2 multiples of 4 channels.
extern "C" int nnis_retention_chunks(const void* q, const void* k, const void* v, int qkv_dtype, int q_stride, int k_stride, int v_stride,
                                     const float* head_decay, const float* rot_cos, const float* rot_sin, int rot_dim, int rot_positions,
                                     const int* tok_pos, float scale, float* state, const int* seq_slot, const int* seq_start, int batch,
                                     int tokens, int heads, int key_dim, int value_dim, float* out, float* scratch, void* stream) {
  NNIS_REQUIRE(nnis_dtype_ok(qkv_dtype), "retention: unknown dtype %d", qkv_dtype);
  NNIS_REQUIRE(nnis_chunked_takes(key_dim, value_dim) && heads > 0 && heads <= 65535 && batch >= 0 && batch <= 65535 && tokens >= 0,
               "retention: %d sequences of %d heads of %d and %d channels are not taken in chunks", batch, heads, key_dim, value_dim);
  NNIS_REQUIRE(q && k && v && head_decay && tok_pos && state && seq_slot && seq_start && out && scratch, "retention: a pointer is missing");
  const uintptr_t quarter = qkv_dtype == NNIS_F32 ? 16 : 8;
  NNIS_REQUIRE(((uintptr_t)q | (uintptr_t)k) % quarter == 0 && q_stride % 4 == 0 && k_stride % 4 == 0 && rot_dim % 8 == 0 && rot_dim <= key_dim &&
                   ((uintptr_t)scratch | (uintptr_t)rot_cos | (uintptr_t)rot_sin) % 16 == 0 && (rot_dim == 0 || (rot_cos && rot_sin && rot_positions > 0)),
               "retention: rows or tables that cannot be loaded four channels at a time");
  if (batch == 0 || tokens == 0) return 0;
  const int chunks = tokens / kChunk + batch;
  RetentionChunkArgs a;
  ChunkArgs& c = a.c;
  c.seq_slot = seq_slot; c.seq_start = seq_start; c.batch = batch; c.heads = heads; c.key_dim = key_dim; c.value_dim = value_dim;
  lay_out(c, scratch, chunks, false);
  c.v = v; c.v_stride = v_stride;
  c.state = state; c.state_row = value_dim; c.state_column = 1; c.out = out;
  a.q = q; a.k = k; a.q_stride = q_stride; a.k_stride = k_stride; a.scale = scale; a.head_decay = head_decay;
  a.rot_cos = rot_cos; a.rot_sin = rot_sin; a.tok_pos = tok_pos; a.rot_dim = rot_dim; a.rot_positions = rot_positions;
  hipStream_t s = (hipStream_t)stream;
  const size_t lds = 2 * kChunk * (size_t)(key_dim + 4) * sizeof(float);
#define NNIS_PREPARE(KT, T)                                                                                                                 \
  NNIS_REQUIRE(hipFuncSetAttribute((const void*)chunk_retention_prepare_kernel<KT, T>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) \
                   == hipSuccess, "retention: %zu bytes of LDS were refused", lds);                                                         \
  hipLaunchKernelGGL((chunk_retention_prepare_kernel<KT, T>), dim3(chunks, heads), dim3(256), lds, s, a)
#define NNIS_RUN(KT)                                                                                                       \
  if (qkv_dtype == NNIS_F32) {                                                                                             \
    NNIS_PREPARE(KT, float);                                                                                               \
    hipLaunchKernelGGL((chunk_scan_kernel<KT, false, float>), dim3(heads, value_dim / 16, batch), dim3(kWave * kScanWaves), 0, s, c);     \
  } else {                                                                                                                 \
    NNIS_PREPARE(KT, bf16_t);                                                                                              \
    hipLaunchKernelGGL((chunk_scan_kernel<KT, false, bf16_t>), dim3(heads, value_dim / 16, batch), dim3(kWave * kScanWaves), 0, s, c);    \
  }
  NNIS_KEY_TILES(NNIS_RUN)
#undef NNIS_RUN
#undef NNIS_PREPARE
  NNIS_LAUNCH_CHECK("retention (chunks)");
  return 0;
}
