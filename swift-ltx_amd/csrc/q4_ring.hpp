// q4_ring.hpp -- pieces shared by the kernels whose operands pass through a
// ring of direct-to-LDS copies (q4_wide.hip, q4_strip.hip).
#pragma once

#include <type_traits>
#include <utility>

#include "q4_common.hpp"

namespace sltx {

typedef __attribute__((address_space(3))) void* lds_ptr_t;

#define RING_LDS_BARRIER() asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory")

// f(integral_constant<int, i>) for i = 0 .. N - 1, unrolled
template <typename F, int... I>
__device__ __forceinline__ void static_for_seq(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_seq(f, std::make_integer_sequence<int, N>{});
}

// LDS reads the compiler does not see as memory operations.  Its wait-count
// pass cannot tell reads of one ring stage from copies in flight into
// another once the loop's back-edge merges its state, and would drain every
// copy in flight (vmcnt(0)) before the first read of each unrolled
// iteration; the stage a round reads has been waited for by that round's
// own vmcnt and barrier.  The results must pass through lds_wait() before
// use.
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(lds_ptr_t)(p);
}
__device__ __forceinline__ u32x4 ds_read16(uint32_t a) {
    u32x4 v;
    asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(a) : "memory");
    return v;
}
__device__ __forceinline__ uint32_t ds_read4(uint32_t a) {
    uint32_t v;
    asm volatile("ds_read_b32 %0, %1" : "=v"(v) : "v"(a) : "memory");
    return v;
}

__device__ __forceinline__ f32x16 mfma32_f16(u32x4 a, u32x4 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

}  // namespace sltx
