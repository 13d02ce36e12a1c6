// Two products of the same up to 16 rows in one launch: gemm_mfma.hip's kernel for few tokens over two packed weights that lie one behind
// the other in whole strips, each product to a place and type of its own.  K is cut, and its parts are added, as there: the same numbers.
// (A file of its own: as a variant of that kernel in its file it moved the others, and steps of 30 rows lost 0.5%.)
#include "product.h"

namespace {

struct TwoOut {
  bf16_t* first;  // [m, columns]
  int columns;
  void* second;   // [m, n - columns]
  int second_f32;
};

// KSPLIT waves share a strip's K, DEPTH chunks of 64 asked for together
template <int KSPLIT>
__global__ __launch_bounds__(KSPLIT > 4 ? 64 * KSPLIT : 256) void gemm_two_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w, TwoOut y, int m,
                                                                                int n, int k) {
  constexpr int kWaves = KSPLIT > 4 ? KSPLIT : 4, DEPTH = 4;
  __shared__ float partial[kWaves][kWave][4];
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave, r = lane % 16, g = lane / 16;
  const int strip = blockIdx.x * (kWaves / KSPLIT) + wave / KSPLIT, part = wave % KSPLIT, chunks = nnis_packed_chunks(k);
  const bool active = strip < (n + 15) / 16;
  f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
  const bf16_t* w_ptr = w + nnis_packed_lane(active ? strip * 16 + r : 0, g, k);
  const bf16_t* x_ptr = x + (size_t)(r < m ? r : m - 1) * k;
  for (int base = part; active && base < chunks; base += KSPLIT * DEPTH) {
    bf16x8 wa[DEPTH][2], xa[DEPTH][2];
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int c = base + d * KSPLIT, at = c * 64 + g * 16 + half * 8;
        wa[d][half] = c < chunks ? load_chunk(w_ptr + (size_t)c * kPackedChunkElems + half * kPackedHalfElems) : zero_chunk();
        xa[d][half] = at + 8 <= k ? load_chunk(x_ptr + at) : zero_chunk();
      }
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
#pragma unroll
      for (int half = 0; half < 2; ++half) acc = mfma(wa[d][half], xa[d][half], acc);
  }
  if constexpr (KSPLIT > 1) {
    if (part != 0) *(f32x4*)partial[wave][lane] = acc;
    __syncthreads();
    if (part != 0) return;
#pragma unroll
    for (int other = 1; other < KSPLIT; ++other) acc += *(const f32x4*)partial[wave + other][lane];
  }
  // lane holds D[weight row 4g + e][token r]: four consecutive outputs of one token
  const int column = strip * 16 + g * 4, rest = n - y.columns, valid = n - column >= 4 ? 4 : n - column;
  if (!active || r >= m || valid <= 0) return;
  if (column < y.columns) store4(y.first, (size_t)r * y.columns + column, acc, valid, true);
  else if (y.second_f32) store4((float*)y.second, (size_t)r * rest + column - y.columns, acc, valid, rest % 4 == 0);
  else store4((bf16_t*)y.second, (size_t)r * rest + column - y.columns, acc, valid, rest % 4 == 0);
}

template <int KSPLIT>
void launch_two(const bf16_t* x, const bf16_t* w, const TwoOut& y, int m, int n, int k, hipStream_t stream) {
  constexpr int kWaves = KSPLIT > 4 ? KSPLIT : 4, kStrips = kWaves / KSPLIT;
  hipLaunchKernelGGL(gemm_two_kernel<KSPLIT>, dim3(((n + 15) / 16 + kStrips - 1) / kStrips), dim3(kWave * kWaves), 0, stream, x, w, y, m, n, k);
}

}  // namespace

// w [n, k]: two packed weights, the first of `columns` rows (whole strips), whose product goes to y in bfloat16, the other's to second in
// second_dtype.  Two short kernels are a launch and a trip to memory more than one: 4 rows of 4,096 channels into 128 and 32 columns
// 6.4 and 6.5 us apart, and whole requests of four sequences through six scans and two gated linear attentions 9,794 us and 9,322.  (A
// large product with 16 columns beside it gained nothing in the gated delta rule: 5,290 and 5,329.)
extern "C" int nnis_gemm_two(const void* x, const void* w, void* y, int columns, void* second, int second_dtype, int m, int n, int k, void* stream_ptr) {
  NNIS_REQUIRE(nnis_dtype_ok(second_dtype), "gemm_two: unknown output dtype %d", second_dtype);
  NNIS_REQUIRE(m > 0 && m <= 16 && columns > 0 && columns % 16 == 0 && columns < n && n < 2048 * 16 && k > 0 && k % 8 == 0,
               "gemm_two: %d rows, %d of %d columns and K=%d are not taken", m, columns, n, k);
  for (const void* p : {x, w, (const void*)y, (const void*)second}) NNIS_REQUIRE(p && (uintptr_t)p % 16 == 0, "gemm_two: operands must be there, 16-byte aligned");
  int split = 1;  // (as skinny_split there)
  while (split < 8 && (k + 63) / 64 > split * 4) split *= 2;
  const TwoOut out = {(bf16_t*)y, columns, second, second_dtype == NNIS_F32};
  const auto launch = split == 8 ? launch_two<8> : split == 4 ? launch_two<4> : split == 2 ? launch_two<2> : launch_two<1>;
  launch((const bf16_t*)x, (const bf16_t*)w, out, m, n, k, (hipStream_t)stream_ptr);
  NNIS_LAUNCH_CHECK("gemm_two");
  return 0;
}
