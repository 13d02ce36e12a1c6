// Loads from memory straight into LDS, which a kernel waits for by counting them itself.
#pragma once

typedef __attribute__((address_space(3))) void* lds_ptr_t;

// waits until no more than N of the wave's loads are in flight
template <int N>
__device__ __forceinline__ void wait_loads_but() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }

// 16 bytes a lane from `offset` bytes behind `base` (the same in every lane, below 4 GiB with `uniform_offset`) to lane * 16
// behind `to`.  A buffer load: of one through a global address the compiler thinks that it may come back out of order with
// every other, and then waits for all reads and loads in flight wherever it needs one of them (32-bit
// tiles that did: a prompt of 509 tokens through a 1.1B model 10.39 -> 9.97 ms).
__device__ __forceinline__ void load_to_lds(const void* base, int offset, int uniform_offset, char* to) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc((void*)base, 0, 0xffffffffu, 0x00027000), (lds_ptr_t)to, 16, offset,
                                           uniform_offset, 0, 0);
}
