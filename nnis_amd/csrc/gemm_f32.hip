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
//  * gemm_f32_few_kernel: few rows of X (a decode step, a short prompt), or too few tiles to fill the chip.  The
//    weight is streamed straight into operand registers; the waves of a block share K and meet in LDS.
//  * gemm_f32_tiled_kernel: tiles of 64, 96 or 128 rows and columns, K in steps of 32 through a ring of stages in LDS.
#include "common.h"

#include <type_traits>

namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((address_space(1))) const void* global_ptr_t;
typedef __attribute__((address_space(3))) void* lds_ptr_t;

template <int N>
__device__ __forceinline__ void wait_loads_but() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

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

// ---- few rows -----------------------------------------------------------------------------------------------------
// A block owns S strips of 16 weight rows and NT tiles of 16 rows of X; its W waves take chunks of 16 k in turn (wave
// w the chunks w, w + W, ..: together they read a row's consecutive memory), up to U of a wave's chunks in flight at
// once.  A wave's last chunks, however many, are one round: every round is a trip to memory.
// HALF (up to 8 rows of X): a strip has 8 weight rows; lanes r < 8 and r >= 8 of a load hold the same rows at k that
// are 16 apart, in both operands, so that of the product D[i][j] the quarters i, j < 8 and i, j >= 8 are the sums
// of two halves of a chunk of 32 k (the other two quarters mean nothing).  Twice as many blocks for a product
// whose strips are few, and no lane loads what another one has.
template <typename XT, int S, int NT, int W, int U, bool HALF>
__global__ __launch_bounds__(64 * W) void gemm_f32_few_kernel(const XT* __restrict__ x, const float* __restrict__ w, void* __restrict__ y,
                                                              int y_dtype, int m, int n, int k) {
  static_assert(!HALF || (S == 1 && NT == 1), "half strips come one at a time");
  constexpr int ROWS = HALF ? 8 : 16, CHUNK = HALF ? 32 : 16;
  __shared__ f32x4 parts[W][S * NT][kWave];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int r = lane % 16, g = lane / 16;
  const int unit = blockIdx.x, row0 = blockIdx.y * NT * 16;
  const int k_lane = HALF ? (r / 8) * 16 + g * 4 : g * 4;  // this lane's first k of a chunk

  // rows beyond the ends read a valid row and are not stored
  const float* w_row[S];
  const XT* x_row[NT];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const int row = (unit * S + s) * ROWS + r % ROWS;
    w_row[s] = w + (size_t)(row < n ? row : n - 1) * k + k_lane;
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

  int c = wave;
  auto round = [&](auto count) {  // this wave's next `count` chunks, none of which reaches beyond K
    constexpr int N = decltype(count)::value;
    f32x4 wv[N][S], xv[N][NT];
#pragma unroll
    for (int u = 0; u < N; ++u) {
#pragma unroll
      for (int s = 0; s < S; ++s) wv[u][s] = load4(w_row[s] + (c + u * W) * CHUNK);
#pragma unroll
      for (int t = 0; t < NT; ++t) xv[u][t] = load4(x_row[t] + (c + u * W) * CHUNK);
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
    for (int t = 0; t < NT; ++t) xv[t] = in ? xv[t] : zero;
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int t = 0; t < NT; ++t) sum[s][t] = multiply16(wv[s], xv[t], sum[s][t]);
  }

#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int t = 0; t < NT; ++t) parts[wave][s * NT + t][lane] = sum[s][t];
  __syncthreads();
  for (int item = wave; item < S * NT; item += W) {  // a wave adds up a (strip, tile)'s parts in their order
    if (HALF && (g >= 2 || r >= 8)) continue;
    f32x4 total = parts[0][item][lane];
    if constexpr (HALF) total += parts[0][item][lane + 40];  // rows and columns 8 on
#pragma unroll
    for (int p = 1; p < W; ++p) {
      total += parts[p][item][lane];
      if constexpr (HALF) total += parts[p][item][lane + 40];
    }
    const int row = row0 + (item % NT) * 16 + r;
    if (row < m) store_columns(y, y_dtype, row, (unit * S + item / NT) * ROWS + g * 4, n, total);
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
template <int BM, int BN, int NS>
__global__ __launch_bounds__(256) void gemm_f32_tiled_kernel(const float* __restrict__ x, const float* __restrict__ w, void* __restrict__ y,
                                                             int y_dtype, int m, int n, int k, int col_blocks) {
  constexpr int TM = BM / 32, TN = BN / 32;  // tiles of 16 x 16 a wave has, each way
  constexpr int A_LOADS = BM / 32, B_LOADS = BN / 32, LOADS = A_LOADS + B_LOADS;  // load instructions a wave and step
  constexpr int A_BYTES = BM * kStepK * 4, STAGE_BYTES = (BM + BN) * kStepK * 4;
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
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
  const float* a_src[A_LOADS];
  const float* b_src[B_LOADS];
#pragma unroll
  for (int o = 0; o < A_LOADS; ++o) {
    const int row = row0 + (o * 4 + wave) * 8 + lane / 8;
    a_src[o] = x + (size_t)(row < m ? row : m - 1) * k;
  }
#pragma unroll
  for (int o = 0; o < B_LOADS; ++o) {
    const int row = col0 + (o * 4 + wave) * 8 + lane / 8;
    b_src[o] = w + (size_t)(row < n ? row : n - 1) * k;
  }
  // Step s lies in stage s % NS.  A step beyond the end, and the last step's chunks beyond K, are asked for from the
  // row's first chunk: valid memory; the former nobody reads, the latter count as zeros.
  const int steps = (k + kStepK - 1) / kStepK;
  auto ask = [&](int step, int stage) {
    char* base = f32_lds + stage * STAGE_BYTES + wave * 1024;
    const int at = step * kStepK + chunk_k;
    const int from = at < k ? at : 0;
#pragma unroll
    for (int o = 0; o < A_LOADS; ++o)
      __builtin_amdgcn_global_load_lds((global_ptr_t)(a_src[o] + from), (lds_ptr_t)(base + o * 4096), 16, 0, 0);
#pragma unroll
    for (int o = 0; o < B_LOADS; ++o)
      __builtin_amdgcn_global_load_lds((global_ptr_t)(b_src[o] + from), (lds_ptr_t)(base + A_BYTES + o * 4096), 16, 0, 0);
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
#pragma unroll
    for (int j = 0; j < TN; ++j)
      store_columns(y, y_dtype, row, col0 + wave_n * (BN / 2) + j * 16 + g * 4, n, total[i][j] + sum[i][j]);
  }
}

template <typename XT, int S, int NT, int W, int U, bool HALF = false>
void launch_few(const void* x, const float* w, void* y, int y_dtype, int m, int n, int k, hipStream_t stream) {
  const int rows = (HALF ? 8 : 16) * S;
  const dim3 grid((n + rows - 1) / rows, (m + 16 * NT - 1) / (16 * NT));
  hipLaunchKernelGGL((gemm_f32_few_kernel<XT, S, NT, W, U, HALF>), grid, dim3(64 * W), 0, stream, (const XT*)x, w, y, y_dtype, m, n, k);
}

template <int BM, int BN, int NS>
int launch_tiled(const float* x, const float* w, void* y, int y_dtype, int m, int n, int k, hipStream_t stream) {
  constexpr int lds = NS * (BM + BN) * kStepK * 4;
  static_assert(lds <= 160 * 1024, "a compute unit has 160 KB");
  auto kernel = gemm_f32_tiled_kernel<BM, BN, NS>;
  NNIS_REQUIRE(hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess,
               "gemm_f32: %d bytes of LDS were refused", lds);
  const int col_blocks = (n + BN - 1) / BN;
  const long long blocks = (long long)col_blocks * ((m + BM - 1) / BM);
  hipLaunchKernelGGL(kernel, dim3((unsigned)blocks), dim3(256), lds, stream, x, w, y, y_dtype, m, n, k, col_blocks);
  return 0;
}

// Which kernel a product takes.  Up to 16 rows the weight's bytes and the trips to memory set the time, measured with 8
// rows over cold weights, microseconds (32-bit; the ordered kernel in brackets): half strips while whole ones leave half
// the compute units without a block, 2048 x 5632 14.0 against 21 (295), 576 x 1536 5.9 against 7.2 (84), but 2560 x 2048 10.1 against
// 8.7; blocks of 4 waves where the strips are many, 11264 x 2048 21.9 against 24.5 (220); two strips a block beyond, 49152 x
// 576 27.7 against 29.1, 32000 x 2048 59.1 against 61.5.  Beyond 16 rows a variant's time is close to its rounds of blocks on 256
// compute units times its blocks' time, which is a slope times K and a start: the least of these is taken.  Measured:
// 64 x 2048 x 2048 14.0 us (two strips, one tile a block), 128 x 2048 x 2048 18.7 (2 x 2), 128 x 11264 x 2048 60 (tiles of 64 x 96; 75
// in 64 x 64), 509 x 2048 x 5632 112 (64 x 64), 4000 x 11264 x 2048 1,443 (128 x 128; 128 TFLOP/s of the instruction's 157).
struct Variant {
  int rows, columns;  // of a block
  float slope, start; // microseconds: slope * K + start for a round of blocks
};
constexpr Variant kVariants[] = {
    {16, 16, 0.0050f, 2.0f}, {16, 32, 0.0064f, 2.0f}, {32, 32, 0.0083f, 2.0f}, {64, 32, 0.0135f, 2.0f},
    {32, 64, 0.0105f, 3.5f}, {64, 64, 0.0189f, 3.5f}, {64, 96, 0.0280f, 3.5f}, {96, 64, 0.0280f, 3.5f}, {96, 96, 0.0405f, 3.5f},
    {64, 128, 0.0365f, 3.5f}, {128, 64, 0.0365f, 3.5f}, {128, 96, 0.0540f, 3.5f}, {128, 128, 0.0700f, 3.5f}};
constexpr int kFewVariants = 4, kCountVariants = sizeof(kVariants) / sizeof(kVariants[0]);
enum : int { kHalfStrips = kCountVariants, kFourWaves, kTwoStrips, kHints };

int pick_variant(bool f32, int m, int n, int k) {
  if (m <= 16) {
    if (m <= 8 && n <= 2048) return kHalfStrips;
    return n <= 8192 ? 0 : (n < 24000 ? kFourWaves : kTwoStrips);
  }
  int best = 0;
  float least = 0.0f;
  for (int v = 0; v < (f32 ? kCountVariants : kFewVariants); ++v) {  // (rows in 16 bits are widened on their way into registers)
    const Variant& it = kVariants[v];
    const long long blocks = (long long)((m + it.rows - 1) / it.rows) * ((n + it.columns - 1) / it.columns);
    const float time = (float)((blocks + 255) / 256) * it.slope * (float)k + it.start;
    if (v == 0 || time < least) {
      best = v;
      least = time;
    }
  }
  return best;
}

}  // namespace

extern "C" int nnis_gemm_f32(const void* x, int x_dtype, const float* w, void* y, int y_dtype, int m, int n, int k, int hint, void* stream) {
  NNIS_REQUIRE(nnis_dtype_ok(x_dtype) && nnis_dtype_ok(y_dtype), "gemm_f32: unknown dtype (x %d, y %d)", x_dtype, y_dtype);
  NNIS_REQUIRE(m >= 0 && n > 0 && k > 0 && k % 4 == 0, "gemm_f32: bad sizes m=%d n=%d k=%d (K a multiple of 4)", m, n, k);
  NNIS_REQUIRE((uintptr_t)x % 16 == 0 && (uintptr_t)w % 16 == 0 && (uintptr_t)y % 16 == 0, "gemm_f32: operands must be 16-byte aligned");
  NNIS_REQUIRE(hint >= -1 && hint < kHints && (hint != kHalfStrips || m <= 8), "gemm_f32: no variant %d for %d rows", hint, m);
  const bool f32 = x_dtype == NNIS_F32;
  const int variant = hint >= 0 ? hint : pick_variant(f32, m, n, k);
  NNIS_REQUIRE(f32 || variant < kFewVariants || variant >= kCountVariants, "gemm_f32: tiles take 32-bit rows");
  NNIS_REQUIRE(variant >= kFewVariants || (m + kVariants[variant].rows - 1) / kVariants[variant].rows <= 65535, "gemm_f32: %d rows exceed the grid limit", m);
  if (m == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
#define NNIS_FEW(...)                                                          \
  if (f32) launch_few<float, __VA_ARGS__>(x, w, y, y_dtype, m, n, k, s);       \
  else launch_few<bf16_t, __VA_ARGS__>(x, w, y, y_dtype, m, n, k, s);          \
  break;
#define NNIS_TILED(...)                                                                \
  if (launch_tiled<__VA_ARGS__>((const float*)x, w, y, y_dtype, m, n, k, s)) return 1; \
  break;
  switch (variant) {  // (strips, tiles, waves, chunks in flight); (rows, columns, stages)
    case 0: NNIS_FEW(1, 1, 8, 4)
    case 1: NNIS_FEW(2, 1, 8, 4)
    case 2: NNIS_FEW(2, 2, 8, 4)
    case 3: NNIS_FEW(2, 4, 4, 2)
    case 4: NNIS_TILED(32, 64, 3)
    case 5: NNIS_TILED(64, 64, 3)
    case 6: NNIS_TILED(64, 96, 3)
    case 7: NNIS_TILED(96, 64, 3)
    case 8: NNIS_TILED(96, 96, 3)
    case 9: NNIS_TILED(64, 128, 3)
    case 10: NNIS_TILED(128, 64, 3)
    case 11: NNIS_TILED(128, 96, 3)
    case 12: NNIS_TILED(128, 128, 2)
    case kHalfStrips: NNIS_FEW(1, 1, 8, 4, true)
    case kFourWaves: NNIS_FEW(1, 1, 4, 8)
    case kTwoStrips: NNIS_FEW(2, 1, 8, 4)
  }
#undef NNIS_FEW
#undef NNIS_TILED
  NNIS_LAUNCH_CHECK("gemm_f32");
  return 0;
}
