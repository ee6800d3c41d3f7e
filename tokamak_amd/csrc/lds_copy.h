#pragma once

// What products share whose operands go from memory to LDS without passing through registers.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#define TK_LDS __attribute__((address_space(3)))

namespace tk {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

union Frag8 {
  u32x4 u;
  bf16x8 v;
};

// f(0), ..., f(N - 1) with the number known to the compiler
template <int I, int N, typename F>
__device__ __forceinline__ void each(const F& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    each<I + 1, N>(f);
  }
}

// 64 lanes' 16 bytes from base + from (a lane's own) to LDS address to, lane after lane.  No register waits for it: the wave's
// count of vector memory operations says when it has come.  ONCE: what nobody else will read (a streaming load).
template <bool ONCE>
__device__ __forceinline__ void copy_to_lds(uint32_t to, uint32_t from, const char* base) {
  if constexpr (ONCE)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(to), "v"(from), "s"(base) : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(from), "s"(base) : "memory", "m0");
}

// The same to LDS address to + AT.
template <int AT>
__device__ __forceinline__ void copy_to_lds_at(uint32_t to, uint32_t from, const char* base) {
  asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(from), "s"(base), "n"(AT) : "memory", "scc", "m0");
}

}  // namespace tk
