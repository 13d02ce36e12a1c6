// How the blocks of one launch hand each other their results (chain.hip, chain_f32.hip).
//
// How words get from block to block: every word of the exchange is kNone (all bits set) before the launch, and is there once it is
// anything else.  Writers store past the caches and never store kNone (a NaN with that payload goes out as another NaN), readers
// load until no word of what they asked for is kNone.  A word carries its own mark, so no order between
// words is needed, no counter and no fence.
//
// Why every wait ends: the stages of a block's operands are blocks of smaller numbers, and a die is handed its blocks in the order
// of their numbers; so the unfinished block with the smallest number is on the chip, or its die is full of blocks of another
// kernel.  Two such launches could fill a die each for the other: those of one process take turns (models/chain.py, in_turn).  Should
// another process's meet one, or a fault keep words away, a wait gives up after kWaitTicks: it says so in `fail` (then all others leave
// too) and in `host_fail`, which the host reads before a step's tokens become the caller's and when a step begins (Engine.check_steps); what was
// not written stays kNone, which is no number, and what hangs on it is none.
#pragma once

#include "common.h"

namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
typedef __attribute__((ext_vector_type(2))) unsigned u32x2;

constexpr unsigned kNone = 0xffffffffu;
constexpr int kPastCaches = 16;              // a buffer access's cache policy: sc1, agent scope
constexpr int kChainHead = 64;               // channels of a head
constexpr int kMostRows = 16;
constexpr int kRunRow = kChainHead + 4;      // words of a run of keys: outputs, reference, sum, two unused
constexpr long long kWaitTicks = 200000000;  // of the 100 MHz clock: 2 s

__device__ __forceinline__ unsigned marked(float v) {
  const unsigned u = __float_as_uint(v);
  return u == kNone ? 0x7fc00000u : u;
}
__device__ __forceinline__ unsigned marked2(bf16_t lo, bf16_t hi) {
  const unsigned u = (unsigned)__builtin_bit_cast(unsigned short, lo) | ((unsigned)__builtin_bit_cast(unsigned short, hi) << 16);
  return u == kNone ? 0x7fc07fc0u : u;
}

__device__ __forceinline__ unsigned pack2(float lo, float hi) {
  typedef __attribute__((ext_vector_type(2))) float f32x2;
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
  return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){lo, hi}, bf16x2));
}
__device__ __forceinline__ unsigned marked2(unsigned packed) { return packed == kNone ? 0x7fc07fc0u : packed; }

// where a lane reads: its own part of a byte offset, and the part that is the wave's
struct At {
  unsigned lane, wave;
};

struct Exchange {
  __amdgpu_buffer_rsrc_t r;
  unsigned *fail, *host_fail;
  bool near;

  template <typename Args>
  __device__ __forceinline__ Exchange(const Args& a, unsigned* words, unsigned bytes, bool near_ = true)
      : r(__builtin_amdgcn_make_buffer_rsrc(words, 0, bytes, 0x00020000)), fail(a.fail), host_fail(a.host_fail), near(near_) {}

  // whether a wait is to be left: every 256th look, by the clock and by what others found
  __device__ __forceinline__ bool leave(int& looks, long long& since) const {
    if ((++looks & 255) != 0) return false;
    const long long now = wall_clock64();
    if (looks == 256) since = now;
    if (__hip_atomic_load(fail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return true;
    if (now - since < kWaitTicks) return false;
    __hip_atomic_store(fail, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(host_fail, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    return true;
  }

  // Until one word of a stage further ahead is there: a block that is on the chip early looks now and then at one word, so that
  // the words of the stage at work are not asked for by every block of the layers behind it.
  template <bool ONE>  // the first wave looks for the whole block
  __device__ __forceinline__ void gate(unsigned word, int wave) const {
    if (!ONE || wave == 0) {
      int looks = 0;
      long long since = 0;
      while (true) {
        const unsigned u = __builtin_amdgcn_raw_buffer_load_b32(r, word * 4, 0, kPastCaches);
        asm volatile("" ::: "memory");  // (asked for anew each time)
        if (__builtin_amdgcn_readfirstlane(u) != kNone || leave(looks, since)) break;
        __builtin_amdgcn_s_sleep(4);
      }
    }
    if (ONE) __syncthreads();
  }

  // 16 bytes a lane N times, and beside each an M-th of 4 or 8 bytes: `ask(i)` gives the i-th's byte offsets, the lane's part and
  // the wave's; whether all of them are there
  template <int POLICY, int N, typename Ask>
  __device__ __forceinline__ bool look(u32x4 (&v)[N], Ask ask) const {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = __builtin_amdgcn_raw_buffer_load_b128(r, ask(i).lane, ask(i).wave, POLICY);
    asm volatile("" ::: "memory");  // (asked for anew each time)
    unsigned top = 0;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) top = max(top, v[i][e]);
    return !__any(top == kNone);
  }
  template <int POLICY, int N, typename Ask, typename T, int M, typename AskBeside>
  __device__ __forceinline__ bool look(u32x4 (&v)[N], Ask ask, T (&w)[M], AskBeside ask_beside) const {
#pragma unroll
    for (int i = 0; i < M; ++i) {
      if constexpr (sizeof(T) == 4) w[i] = __builtin_amdgcn_raw_buffer_load_b32(r, ask_beside(i).lane, ask_beside(i).wave, POLICY);
      else w[i] = __builtin_amdgcn_raw_buffer_load_b64(r, ask_beside(i).lane, ask_beside(i).wave, POLICY);
    }
    const bool all = look<POLICY>(v, ask);
    unsigned top = 0;
#pragma unroll
    for (int i = 0; i < M; ++i) {
      if constexpr (sizeof(T) == 4) top = max(top, w[i]);
      else top = max(top, max(w[i][0], w[i][1]));
    }
    return !__any(top == kNone) && all;
  }

  // ... until all of them are there.  The first look goes through the caches, which may have them from a neighbour's: a word is
  // written once in a launch, so a cached one is what was written or still none; a line that was fetched half written stays
  // so, and all further looks go past them.  (16 rows of 32 heads and a width of 2,048 1,405 us and 1,259, 8 rows 1,147 and 1,112; a
  // prompt of 177 rows of width 576, with nothing through the caches 552 and 482.  `near`: few rows of narrow models leave it out.)
  template <int N, typename... Rest>
  __device__ __forceinline__ void take(u32x4 (&v)[N], Rest&&... rest) const {
    if (near && look<0>(v, rest...)) return;
    int looks = 0;
    long long since = 0;
    while (!look<kPastCaches>(v, rest...) && !leave(looks, since)) {}
  }
  __device__ __forceinline__ void put(unsigned word, unsigned v) const { __builtin_amdgcn_raw_buffer_store_b32(v, r, word * 4, 0, kPastCaches); }
  __device__ __forceinline__ void put(unsigned word, u32x2 v) const { __builtin_amdgcn_raw_buffer_store_b64(v, r, word * 4, 0, kPastCaches); }
  __device__ __forceinline__ void put(unsigned word, u32x4 v) const { __builtin_amdgcn_raw_buffer_store_b128(v, r, word * 4, 0, kPastCaches); }
};

// words that a strip of the stream has for its rows' parts of their sums of squares
__host__ __device__ constexpr int sum_words(int rows) { return rows <= 4 ? 4 : rows <= 8 ? 8 : 16; }

// What stands between a stage's last operand and its words is a chain of instructions of one wave, four cycles each and more: the
// ends of the products are kept short (lanes meet by the register moves of common.h).

// Which of a result's elements (16 channels of up to 16 rows) a lane ends.  The matrix instruction leaves a lane four channels of a row;
// of up to 8 and 4 rows half and three quarters of the lanes would have none, and from LDS each takes two or one.
template <int ROWS>
struct Ends {
  static constexpr int kEach = ROWS <= 4 ? 1 : ROWS <= 8 ? 2 : 4;
  int row, first, from;  // the first of its channels; the lane that had them
  __device__ __forceinline__ explicit Ends(int lane)
      : row(lane % 16 / (4 / kEach)), first(lane / 16 * 4 + lane % (4 / kEach) * kEach), from(lane / 16 * 16 + row) {}
};
template <int N>
struct Floats {
  float v[N];
  __device__ __forceinline__ float& operator[](int e) { return v[e]; }
  __device__ __forceinline__ float operator[](int e) const { return v[e]; }
};
template <int N>
__device__ __forceinline__ Floats<N> load_floats(const float* p) {
  typedef __attribute__((ext_vector_type(2))) float f32x2;
  Floats<N> out;
  if constexpr (N == 4) {
    const f32x4 v = *(const f32x4*)p;
#pragma unroll
    for (int e = 0; e < 4; ++e) out[e] = v[e];
  } else if constexpr (N == 2) {
    const f32x2 v = *(const f32x2*)p;
    out[0] = v[0];
    out[1] = v[1];
  } else {
    out[0] = *p;
  }
  return out;
}
template <int N>
__device__ __forceinline__ void put_floats(const Exchange& ex, unsigned word, const Floats<N>& v) {
  if constexpr (N == 4) ex.put(word, (u32x4){marked(v[0]), marked(v[1]), marked(v[2]), marked(v[3])});
  else if constexpr (N == 2) ex.put(word, (u32x2){marked(v[0]), marked(v[1])});
  else ex.put(word, marked(v[0]));
}

// The scales of up to ROWS rows that a norm prepared, by one wave of a block beside its products: the parts of a row's sum of squares lie behind
// each of the stream's strips (up to 64 of them), and are added up strip 4 c + g by strip in lane group g, then over the groups.
template <int ROWS>
struct RowScales {
  static constexpr int kFours = sum_words(ROWS) / 4;  // 16 bytes that a strip has of them: loads of the wave
  __attribute__((aligned(16))) unsigned parts[kFours * kWave * 4];  // [strip][row]
  float scale[16];

  // where load i of a lane is, from the first strip's sums on; `stride`: bytes from strip to strip
  static __device__ __forceinline__ At at(int i, int lane, unsigned first_word, unsigned stride, int strips) {
    const int n = i * kWave + lane;
    return At{(first_word + n % kFours * 4) * 4 + min(n / kFours, strips - 1) * stride, 0};
  }
  __device__ __forceinline__ void make(const u32x4 (&got)[kFours], int lane, int strips, float inv_width, float eps) {
#pragma unroll
    for (int i = 0; i < kFours; ++i) *(u32x4*)&parts[(i * kWave + lane) * 4] = (i * kWave + lane) / kFours < strips ? got[i] : (u32x4){0, 0, 0, 0};
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // (all sixteen, zeros beyond the strips: told to stop there, the compiler goes through its registers in a loop, 0.2 us)
    float part[16], sum = 0.0f;
#pragma unroll
    for (int c = 0; c < 16; ++c) part[c] = __uint_as_float(parts[(4 * c + lane / 16) * sum_words(ROWS) + lane % sum_words(ROWS)]);
#pragma unroll
    for (int c = 0; c < 16; ++c) sum += part[c];
    sum = sum_32_apart(sum_16_apart(sum));
    if (lane < sum_words(ROWS)) scale[lane] = 1.0f / sqrtf(sum * inv_width + eps);
  }
};

__global__ __launch_bounds__(256) void chain_clear_kernel(u32x4* words, unsigned n, u32x4* runs, unsigned n_runs, unsigned* fail) {
  for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < n + n_runs; i += gridDim.x * 256) {
    u32x4* at = i < n ? words + i : runs + (i - n);
    *at = (u32x4){kNone, kNone, kNone, kNone};
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) *fail = 0;
}

inline int chain_clear(void* words, long long word_count, void* runs, long long run_count, unsigned* fail, hipStream_t stream) {
  const unsigned fours = (unsigned)(word_count / 4), run_fours = (unsigned)(run_count / 4), blocks = (fours + run_fours + 255) / 256;
  hipLaunchKernelGGL(chain_clear_kernel, dim3(blocks < 1024 ? blocks : 1024), dim3(256), 0, stream, (u32x4*)words, fours, (u32x4*)runs, run_fours, fail);
  NNIS_LAUNCH_CHECK("chain_clear");
  return 0;
}

}  // namespace
