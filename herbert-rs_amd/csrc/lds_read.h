// Reads of LDS by hand, for kernels whose matrix products follow each other faster than the compiler's waits let them.
#pragma once
#include "common.h"
#include <type_traits>

typedef __bf16 hb_bf16x8 __attribute__((ext_vector_type(8)));

// A read of 16 bytes from LDS that the compiler does not follow: it neither waits for it nor
// knows that it is in flight, so the caller waits by count (lds_wait<N>: at most N reads, in the
// order in which they were issued, may still be on their way) before the value is used. The
// compiler's own waits drain every read in flight (lgkmcnt(0)) each time a value is needed, the
// one issued a moment ago included (and, before any read of LDS, every load on its way into LDS, whichever
// stage it fills); with three reads ahead of their products a wave of the prompt attention then stood still for a read's whole way through LDS eleven times a page.
template <int BYTES_ON>
__device__ __forceinline__ hb_bf16x8 lds_read_ahead(const void* p) {
    hb_bf16x8 v;
    const uint32_t at = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)p;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(at), "n"(BYTES_ON));
    return v;
}
// (the value that is about to be used goes through the wait, so that its use cannot be moved before it)
template <int N>
__device__ __forceinline__ void lds_wait(hb_bf16x8& arrived) {
    asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(arrived) : "n"(N));
}

// f(integral_constant<int, B>), ..., f(integral_constant<int, E - 1>): a loop whose index is a
// constant inside the body
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}
