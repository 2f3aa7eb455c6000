// Float32 products on the bfloat16 matrix cores. A float32 number is the sum of three bfloat16 ones, exactly: v rounded to
// bfloat16, the rest rounded, and what then is left, which has at most eight bits. Of the nine products of two such
// numbers' parts six are summed (the other three are below 2^-25 of the whole product), each exact: a product of
// 16 x 16 x 32 costs six instructions of 16 cycles where the float32 matrix instructions need eight of 32, three
// where one side is stored in bfloat16. The leading parts' products and the five smaller ones have a sum each: the matrix cores round a
// sum once in 32 k, and the smaller sums' roundings weigh next to nothing. Over normal, positive and very uneven operands and K from
// 32 to 12288 the error against 64 bits is 0.32 to 0.94 of that of a chain of fmaf in the same stretches, normal operands and K = 4 0.68, 16 0.44 (all six in one sum: 0.36 to 0.92, with a drift
// towards -infinity that the matrix cores' own adding brings and the short sums here do not show).
// What is not finite spoils its parts (infinity minus infinity), as does what lies beyond 2^112 or sums beyond 2^96: callers take a sum that is
// not finite from `mend_blocks` instead.
#pragma once
#include "mfma_f32.h"

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// Eight neighbouring elements of a row as they are stored, and their parts. A lane's eight are those of row lane % 16 at
// k0 + 8 (lane / 16): what a product of 16 x 16 x 32 wants of either operand.
template <class T> struct Oct;
template <> struct Oct<float> {
    f32x4 quad[2];
};
template <> struct Oct<bf16> {
    bf16x8 all;
};
template <class T> struct Parts {
    static constexpr int COUNT = sizeof(T) == 4 ? 3 : 1;
    bf16x8 part[COUNT];
};

// How eight elements are loaded: element by element; float32 16 and bfloat16 8 bytes at a time (rows on such borders, K a multiple of 4); either
// 16 bytes at a time (K a multiple of 8 where bfloat16 is concerned).
enum { OCT_SINGLE, OCT_HALVES, OCT_WHOLE };
// The eight of `row` from k on. Of vector loads, what lies at or beyond K is something of the row's: `ends` makes zeros of it. No branch hangs on
// k, so that no load is waited for where the paths of one would meet. Element by element: zeros from K on.
template <int HOW>
__device__ __forceinline__ Oct<float> load_oct(const float* row, int k, int K) {
    if (HOW != OCT_SINGLE) return Oct<float>{{*(const f32x4*)(row + (k < K ? k : 0)), *(const f32x4*)(row + (k + 4 < K ? k + 4 : 0))}};
    return Oct<float>{{load_quad<false>(row + k, K - k), load_quad<false>(row + k + 4, K - k - 4)}};
}
__device__ __forceinline__ Oct<bf16> two_halves(const bf16* first, const bf16* second) {
    const uint2 halves[2] = {*(const uint2*)first, *(const uint2*)second};
    return __builtin_bit_cast(Oct<bf16>, halves);
}
template <int HOW>
__device__ __forceinline__ Oct<bf16> load_oct(const bf16* row, int k, int K) {
    if (HOW == OCT_WHOLE) return Oct<bf16>{*(const bf16x8*)(row + (k < K ? k : 0))};
    if (HOW == OCT_HALVES) return two_halves(row + (k < K ? k : 0), row + (k + 4 < K ? k + 4 : 0));
    Oct<bf16> r;
#pragma unroll
    for (int i = 0; i < 8; ++i) r.all[i] = k + i < K ? __builtin_bit_cast(__bf16, row[k + i].bits) : (__bf16)0.f;
    return r;
}
// The eight at `offset` elements from a place that is the same for all lanes.
template <int HOW>
__device__ __forceinline__ Oct<float> load_oct(const float* place, unsigned offset) {
    const char* at = (const char*)place + offset * 4u;
    return Oct<float>{{*(const f32x4*)at, *(const f32x4*)(at + 16)}};
}
template <int HOW>
__device__ __forceinline__ Oct<bf16> load_oct(const bf16* place, unsigned offset) {
    const bf16* at = (const bf16*)((const char*)place + offset * 2u);
    return HOW == OCT_WHOLE ? Oct<bf16>{*(const bf16x8*)at} : two_halves(at, at + 4);
}
__device__ __forceinline__ void ends(Oct<float>& o, int left) {
#pragma unroll
    for (int i = 0; i < 8; ++i) o.quad[i / 4][i % 4] = i < left ? o.quad[i / 4][i % 4] : 0.f;
}
__device__ __forceinline__ void ends(Oct<bf16>& o, int left) {
#pragma unroll
    for (int i = 0; i < 8; ++i) o.all[i] = i < left ? o.all[i] : (__bf16)0.f;
}

// A float32 number's parts are those of 2^16 times it: what it has below 2^-133, where bfloat16 ends, is not lost then, down to float32's own last
// bit. (Operands of 1e-38 and 10: an error of 2.7e-3 without, 1.3e-7 so. It costs a product of few rows a tenth, float32 weights, 2 x 2048 x 2048 9.5 ->
// 10.5 us, a tile 0 to 3 %.)
#define SPLIT_SCALE 65536.f
// Each rest, v - (float)part, is exact and one instruction: a product of two pairs and a sum, with -1 and 0. (The pair -1, 0 is hidden
// from the compiler, which would write the float -1, whose halves are 0, -1, in its place.)
__device__ __forceinline__ void split_pair(float v0, float v1, bf16x2& top, bf16x2& mid, bf16x2& low) {
    unsigned first_bits = 0x0000bf80u, second_bits = 0xbf800000u;
    asm("" : "+s"(first_bits), "+s"(second_bits));
    const bf16x2 first = __builtin_bit_cast(bf16x2, first_bits), second = __builtin_bit_cast(bf16x2, second_bits);
    top = bf16x2{(__bf16)v0, (__bf16)v1};
    v0 = __builtin_amdgcn_fdot2_f32_bf16(top, first, v0, false), v1 = __builtin_amdgcn_fdot2_f32_bf16(top, second, v1, false);
    mid = bf16x2{(__bf16)v0, (__bf16)v1};
    v0 = __builtin_amdgcn_fdot2_f32_bf16(mid, first, v0, false), v1 = __builtin_amdgcn_fdot2_f32_bf16(mid, second, v1, false);
    low = bf16x2{(__bf16)v0, (__bf16)v1};
}
__device__ __forceinline__ Parts<float> split(const Oct<float>& o) {
    Parts<float> r;
#pragma unroll
    for (int i = 0; i < 8; i += 2) {
        bf16x2 top, mid, low;
        split_pair(o.quad[i / 4][i % 4] * SPLIT_SCALE, o.quad[i / 4][i % 4 + 1] * SPLIT_SCALE, top, mid, low);
        r.part[0][i] = top[0], r.part[0][i + 1] = top[1];
        r.part[1][i] = mid[0], r.part[1][i + 1] = mid[1];
        r.part[2][i] = low[0], r.part[2][i + 1] = low[1];
    }
    return r;
}
__device__ __forceinline__ Parts<bf16> split(const Oct<bf16>& o) { return Parts<bf16>{{o.all}}; }

// What sums of products of such parts are multiplied by, in the end.
template <class TW, class TA>
__device__ __forceinline__ constexpr float split_unit() {
    return (Parts<TW>::COUNT == 3 ? 1.f / SPLIT_SCALE : 1.f) * (Parts<TA>::COUNT == 3 ? 1.f / SPLIT_SCALE : 1.f);
}

// Which parts meet, the smallest products first; the last one has the sum `top`, the others `low`.
#define SPLIT_PRODUCTS 6
template <int W_PARTS, int A_PARTS>
struct SplitOrder {
    static constexpr int w[SPLIT_PRODUCTS] = {0, 2, 1, 0, 1, 0}, a[SPLIT_PRODUCTS] = {2, 0, 1, 1, 0, 0};
    static constexpr bool there(int p) { return w[p] < W_PARTS && a[p] < A_PARTS; }
};
__device__ __forceinline__ f32x4 mfma_k32(bf16x8 w, bf16x8 a, f32x4 sums) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, a, sums, 0, 0, 0);
}
// One 16 x 16 x 32 product; a lane's four sums are those of mfma_k4.
template <class TW, class TA>
__device__ __forceinline__ void mfma_split(const Parts<TW>& w, const Parts<TA>& a, f32x4& top, f32x4& low) {
    typedef SplitOrder<Parts<TW>::COUNT, Parts<TA>::COUNT> order;
#pragma unroll
    for (int p = 0; p < SPLIT_PRODUCTS; ++p)
        if (order::there(p)) {
            f32x4& sums = p == SPLIT_PRODUCTS - 1 ? top : low;
            sums = mfma_k32(w.part[order::w[p] % Parts<TW>::COUNT], a.part[order::a[p] % Parts<TA>::COUNT], sums);
        }
}

// The sum of one output in plain float32: a chain of fmaf over each stretch of `block` elements of k, the stretches' sums
// one after another.
template <class TA, class TW>
__device__ __forceinline__ float hb_sum_in_order(const TA* a, const TW* w, int K, int block) {
    float total = 0.f;
    for (int k0 = 0; k0 < K; k0 += block) {
        const int end = K - k0 < block ? K : k0 + block;
        float sum = 0.f;
        int k = k0;
#pragma unroll 1
        for (; k + 8 <= end; k += 8) {
            float x[8], y[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = hb_to_float(w[k + i]), y[i] = hb_to_float(a[k + i]);
#pragma unroll
            for (int i = 0; i < 8; ++i) sum = fmaf(x[i], y[i], sum);
        }
#pragma unroll 1
        for (; k < end; ++k) sum = fmaf(hb_to_float(w[k]), hb_to_float(a[k]), sum);
        total += sum;
    }
    return total;
}

__device__ __forceinline__ bool hb_wild(float v) { return !(fabsf(v) < INFINITY); }
__device__ __forceinline__ bool hb_wild(f32x4 v) { return hb_wild(v[0]) || hb_wild(v[1]) || hb_wild(v[2]) || hb_wild(v[3]); }

// Sums of a 16 x 16 block that are not finite, as plain float32 has them; all of a wave calls this. row_of(i): the block's i-th row of A, null
// beyond the last; W: its first row, `columns` of them. A row of A with a NaN is NaN throughout. In others what is not finite
// among the operands says what the sum is, whatever its order, and only sums of finite numbers (parts or sums beyond the range) are
// summed again in their order. A wave looks at 64 elements of a row at a time. A product of 8 rows with 2048 x 2048 float32 weights, 11.3 us, takes 13.2
// where a row is NaN, 53 where one holds an infinity and 92 where one holds 3.4e38 (an output a lane, an element at a time: 504); of
// 512 rows, 4096 x 4096, 124, 127, 338 and 532 us (2,322). (Sixteen columns at a time: 42 and 270 us with an infinity, but registers that cost
// the tiles of 64 x 64 one of two workgroups a CU.)
template <class TA, class TW, class Rows>
__device__ __forceinline__ void mend_block(Rows row_of, const TW* W, size_t ldw, int columns, int K, int block, f32x4& sums) {
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
    const unsigned long long wrong = __ballot(hb_wild(sums));
#pragma unroll 1
    for (int i = 0; i < 16; ++i) {
        const TA* a = row_of(i);
        if (!(wrong >> i & 0x0001000100010001ull) || !a) continue;
        bool none = false;
        for (int k = lane; k < K; k += 8 * HB_WAVE) {
            float y[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) y[u] = hb_to_float(a[k + HB_WAVE * u < K ? k + HB_WAVE * u : k]);
#pragma unroll
            for (int u = 0; u < 8; ++u) none |= y[u] != y[u];
        }
        float value = NAN;
        if (!__any(none)) {
            unsigned nan_or_up = 0, down = 0;                // a bit a column; +infinity in the upper half
#pragma unroll 1
            for (int n0 = 0; n0 < 16; n0 += 4) {             // (four columns at a time: the tiles' registers are not to grow for this)
                const TW* w[4];
#pragma unroll
                for (int n = 0; n < 4; ++n) w[n] = W + (n0 + n < columns ? n0 + n : 0) * ldw;
#pragma unroll 2
                for (int k = lane; k < K; k += HB_WAVE) {
                    const float y = hb_to_float(a[k]);
                    float x[4];
#pragma unroll
                    for (int n = 0; n < 4; ++n) x[n] = hb_to_float(w[n][k]);
#pragma unroll
                    for (int n = 0; n < 4; ++n)
                        if (hb_wild(x[n]) || hb_wild(y)) {
                            const float p = x[n] * y;
                            nan_or_up |= (p != p ? 1u : p > 0.f ? 0x10000u : 0u) << (n0 + n);
                            down |= (p < 0.f ? 1u : 0u) << (n0 + n);
                        }
                }
            }
#pragma unroll
            for (int off = 1; off < HB_WAVE; off <<= 1) nan_or_up |= __shfl_xor(nan_or_up, off, HB_WAVE), down |= __shfl_xor(down, off, HB_WAVE);
            const unsigned nan = nan_or_up | (nan_or_up >> 16 & down), up = nan_or_up >> 16, settled = (nan | up | down) & 0xffffu;
            bool chain = false;
#pragma unroll
            for (int e = 0; e < 4; ++e) chain |= r == i && 4 * q + e < columns && hb_wild(sums[e]) && !(settled >> (4 * q + e) & 1);
            value = nan >> r & 1 ? NAN : up >> r & 1 ? INFINITY : -INFINITY;
            if (__any(chain) && !(settled >> r & 1)) value = hb_sum_in_order(a, W + (size_t)(r < columns ? r : 0) * ldw, K, block);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float v = __shfl(value, 4 * q + e, HB_WAVE);
            if (r == i && hb_wild(sums[e])) sums[e] = v;
        }
    }
}

// The sums of parts' products as the operands' own, all of a wave's blocks: W's row n0 + 16 j is the first of the blocks [j][..], row_of(16 i) that of the blocks [..][i].
template <class TA, class TW, int NB, int MB, class Rows>
__device__ __forceinline__ void mend_blocks(Rows row_of, const TW* W, size_t ldw, int n0, int N, int K, int block, f32x4 (&sums)[NB][MB]) {
    bool wild = false;
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int i = 0; i < MB; ++i) wild |= hb_wild(sums[j][i]), sums[j][i] *= split_unit<TW, TA>();
    if (!__any(wild)) return;
#pragma unroll 1
    for (int b = 0; b < NB * MB; ++b) {                      // (one copy of the code: the block is picked out and put back)
        f32x4 s = sums[0][0];
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int i = 0; i < MB; ++i) s = j * MB + i == b ? sums[j][i] : s;
        const int n = n0 + 16 * (b / MB);
        if (n < N) mend_block<TA, TW>([&](int i) { return row_of(16 * (b % MB) + i); }, W + (size_t)n * ldw, ldw, N - n, K, block, s);
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int i = 0; i < MB; ++i) sums[j][i] = j * MB + i == b ? s : sums[j][i];
    }
}

// Elements of k that are summed from zero; a multiple of every kernel's stage.
#define SPLIT_STRETCH 512
// Pieces of 32 k that are asked for at once where a stretch is not whole.
#define WAVE_DEPTH 4

// A wave's sums over the stretch of k that starts at k0, for NB blocks of 16 rows of W and MB of A (w_row, a_row: the lane's own rows,
// vectors at a time, HOW; q = lane / 16). AHEAD pieces of 32 k of W and A_AHEAD of A are in flight.
template <int AHEAD, int A_AHEAD, int HOW = OCT_WHOLE, class TW, class TA, int NB, int MB>
__device__ __forceinline__ void sum_stretch(const TW* const (&w_row)[NB], const TA* const (&a_row)[MB], int k0, int K, int q,
                                            f32x4 (&top)[NB][MB], f32x4 (&low)[NB][MB]) {
    constexpr int UNITS = SPLIT_STRETCH / 32;
    if (k0 + SPLIT_STRETCH <= K) {
        Oct<TW> w[AHEAD][NB];
        Oct<TA> a[A_AHEAD][MB];
        auto fetch_w = [&](int u) {
#pragma unroll
            for (int j = 0; j < NB; ++j) w[u % AHEAD][j] = load_oct<HOW>(w_row[j] + k0 + 32 * u, 8u * q);
        };
        auto fetch_a = [&](int u) {
#pragma unroll
            for (int i = 0; i < MB; ++i) a[u % A_AHEAD][i] = load_oct<HOW>(a_row[i] + k0 + 32 * u, 8u * q);
        };
#pragma unroll
        for (int u = 0; u < A_AHEAD; ++u) fetch_a(u);
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) fetch_w(u);
        __builtin_amdgcn_sched_barrier(0);           // (no load waits for the sums before it)
#pragma unroll
        for (int u = 0; u < UNITS; ++u) {
            Parts<TW> w_parts[NB];
#pragma unroll
            for (int j = 0; j < NB; ++j) w_parts[j] = split(w[u % AHEAD][j]);
            if (u + AHEAD < UNITS) fetch_w(u + AHEAD);
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                const Parts<TA> a_parts = split(a[u % A_AHEAD][i]);
#pragma unroll
                for (int j = 0; j < NB; ++j) mfma_split<TW, TA>(w_parts[j], a_parts, top[j][i], low[j][i]);
            }
            if (u + A_AHEAD < UNITS) fetch_a(u + A_AHEAD);
        }
        return;
    }
    for (int k = k0; k < K; k += 32 * WAVE_DEPTH) {          // (what is left of k)
        Oct<TW> w[WAVE_DEPTH][NB];
        Oct<TA> a[WAVE_DEPTH][MB];
#pragma unroll
        for (int d = 0; d < WAVE_DEPTH; ++d) {
#pragma unroll
            for (int j = 0; j < NB; ++j) w[d][j] = load_oct<HOW>(w_row[j], k + 32 * d + 8 * q, K);
#pragma unroll
            for (int i = 0; i < MB; ++i) a[d][i] = load_oct<HOW>(a_row[i], k + 32 * d + 8 * q, K);
        }
#pragma unroll
        for (int d = 0; d < WAVE_DEPTH; ++d) {
            const int left = K - k - 32 * d;
            if (left <= 0) break;
            Parts<TW> w_parts[NB];
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                if (left < 32) ends(w[d][j], left - 8 * q);
                w_parts[j] = split(w[d][j]);
            }
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                if (left < 32) ends(a[d][i], left - 8 * q);
                const Parts<TA> a_parts = split(a[d][i]);
#pragma unroll
                for (int j = 0; j < NB; ++j) mfma_split<TW, TA>(w_parts[j], a_parts, top[j][i], low[j][i]);
            }
        }
    }
}
