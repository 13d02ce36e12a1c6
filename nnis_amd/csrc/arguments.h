// The arguments of a launch of one or a few rows, asked for at once.
//
// Arguments lie in memory, and the compiler asks for each where it is first used: a kernel whose arguments fill three lines of 64 bytes makes
// a trip to memory for each of them in turn, in the middle of its own chain of trips.  With a word of each line first, microseconds: the rotation
// of one token 4.4 -> 4.05, a step of 8 heads of 128 x 256 of matrix state 4.2 -> 3.9; kernels whose arguments are one or two lines gain nothing.
#pragma once

#include "common.h"

// 0, once a word of every line is there (what is asked for later is in the scalar cache): added to the index that the kernel's loads begin with
template <typename Args>
__device__ __forceinline__ int arguments_there(const Args& args) {
  static_assert(sizeof(Args) > 64 && sizeof(Args) <= 256, "two to four lines");
  const unsigned* words = (const unsigned*)&args;
  constexpr int kLast = (int)(sizeof(Args) / 4) - 1;
  int zero;
  asm("s_mov_b32 %0, 0" : "=s"(zero) : "s"(words[0]), "s"(words[kLast < 16 ? kLast : 16]), "s"(words[kLast < 32 ? kLast : 32]), "s"(words[kLast]));
  return zero;
}
