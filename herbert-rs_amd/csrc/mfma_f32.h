// Pieces of the kernels that take float32 sums to the matrix cores: the 16 x 16 x 4 product, whose sums keep the order and
// the rounding of a chain of fmaf over ascending k, and how four neighbouring elements of a row reach the lanes it wants.
#pragma once
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

// One 16 x 16 x 4 product: w is W[n = lane % 16, k], a is A[m = lane % 16, k], both for k = k0 + lane / 16; lane l's
// four sums are those of n = 4 (l / 16) .. + 3 and m = l % 16.
__device__ __forceinline__ f32x4 mfma_k4(float w, float a, f32x4 sums) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(w, a, sums, 0, 0, 0);
}

// Four neighbouring elements of a row as float32 (16 or 8 bytes, aligned), or what lies below `left` of them.
template <bool VEC>
__device__ __forceinline__ f32x4 load_quad(const float* p, int left) {
    f32x4 r = {0.f, 0.f, 0.f, 0.f};
    if (VEC) {
        if (left > 0) r = *(const f32x4*)p;
        return r;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (i < left) r[i] = p[i];
    return r;
}
template <bool VEC>
__device__ __forceinline__ f32x4 load_quad(const bf16* p, int left) {
    f32x4 r = {0.f, 0.f, 0.f, 0.f};
    if (VEC) {
        if (left > 0) {
            const uint2 u = *(const uint2*)p;
            r[0] = __uint_as_float(u.x << 16), r[1] = __uint_as_float(u.x & 0xffff0000u);
            r[2] = __uint_as_float(u.y << 16), r[3] = __uint_as_float(u.y & 0xffff0000u);
        }
        return r;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (i < left) r[i] = hb_to_float(p[i]);
    return r;
}

// Four quads, one a lane row of 16 (lane / 16), transposed in registers: x[i] of lane row q was element 4 q + i of 16
// and becomes element 4 i + q, which is what the i-th of four products wants of that lane row.
__device__ __forceinline__ void transpose_quads(f32x4& x) {
    typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
    auto halves = [](float& a, float& b) {
        const u32x2 t = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        a = __uint_as_float(t[0]), b = __uint_as_float(t[1]);
    };
    auto rows = [](float& a, float& b) {
        const u32x2 t = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        a = __uint_as_float(t[0]), b = __uint_as_float(t[1]);
    };
    float x0 = x[0], x1 = x[1], x2 = x[2], x3 = x[3];
    halves(x0, x2);
    halves(x1, x3);
    rows(x0, x1);
    rows(x2, x3);
    x[0] = x0, x[1] = x1, x[2] = x2, x[3] = x3;
}

