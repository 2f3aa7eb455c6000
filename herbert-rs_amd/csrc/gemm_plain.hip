// Matrix product in float32 arithmetic for any storage types and any sizes:
//   C[m, n] (+)= sum_k A[m, k] * W[n, k]      (weights are [out, in], k contiguous)
// It is the whole matrix path of the float32 mode and the fallback of the bfloat16
// mode for shapes its own MFMA kernels refuse. Each output is summed in stretches of K_BLOCK
// elements of k: a stretch from zero over k ascending in blocks of 32 by the split products of mfma_split.h, then the
// stretches' sums one after another. Stretches and blocks lie at fixed places and a block's products come in one order, so an output's value does
// not depend on M, on the tile or kernel it falls in, or on what else is in the batch, and yet
// a product of few rows can give every stretch a wave of its own. (The float32 matrix instructions in the
// same stretches, which this replaced, were further from 64 bits: at K = 2048 4.1e-7 of the sums' root mean square, now 1.3e-7; at
// K = 8704 4.1e-7 and 1.5e-7.)
// In xigh/herbert-rs: crates/backends/backend_bf16/src/kernels.rs:154-164 (float32 sums over k ascending of
// x[m, k] * float(w[n, k]), no bias); crates/backends/backend_vulkan/shaders/bf16_matmul.comp:31-60.
#include "common.h"
#include "mfma_split.h"
#include <type_traits>

HB_MODULE_ERROR_SLOT()

#define K_BLOCK SPLIT_STRETCH

// What a product may do to a sum before it stores it: nothing (rate null), or turn the pre-activation of a
// decay into the decay itself, exp(-exp(rate[n / D]) * softplus(sum + bias[n])) for column n (float32; the
// arithmetic of hb_channel_decay, which does the same to rows that lie in memory). A decay of the other kind
// (rate == bias, the mark of it): sigmoid(sum + bias[n])^root = exp(-root * softplus(-(sum + bias[n]))).
struct DecayEpilogue {
    const float* rate;
    const float* bias;
    int D;
    float root;
    int from;                 // of a batch: the first product that it is for
};

__device__ __forceinline__ float decay_of(const DecayEpilogue& ep, float sum, int n) {
    const float a = sum + ep.bias[n];
    if (ep.rate == ep.bias) {
        const float softplus = -a > 20.f ? -a : log1pf(expf(-a));
        return expf(-ep.root * softplus);
    }
    const float softplus = a > 20.f ? a : log1pf(expf(a));
    return expf(-expf(ep.rate[n / ep.D]) * softplus);
}

// What a lane holds of one output column's four neighbouring rows n .. n + 3 into C[m, n ..].
template <class TC, bool ACCUM, bool VEC>
__device__ __forceinline__ void store_quad(TC* C, int ldc, int m, int n, int N, f32x4 sums, const DecayEpilogue& ep) {
    TC* out = C + (size_t)m * ldc + n;
    if (ep.rate) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (n + e < N) sums[e] = decay_of(ep, sums[e], n + e);
    }
    if (VEC && sizeof(TC) == 4) {
        if (n >= N) return;
        f32x4* o = (f32x4*)out;
        if (ACCUM) sums += *o;
        *o = sums;
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if (n + e >= N) return;
        out[e] = hb_from_float<TC>(ACCUM ? hb_to_float(out[e]) + sums[e] : sums[e]);
    }
}

// The rows of A from m0 on for mend_blocks.
template <class TA>
__device__ __forceinline__ auto rows_of(const TA* A, int lda, int m0, int M) {
    return [=](int i) { return m0 + i < M ? A + (size_t)(m0 + i) * lda : nullptr; };
}

// blockIdx.z: one of a batch of products whose operands lie batch_* elements apart (either way: a pair's lie where they lie).
template <class TA, class TW, class TC>
__device__ __forceinline__ void to_product(const TA* __restrict__& A, const TW* __restrict__& W, TC* __restrict__& C, ptrdiff_t batch_a, ptrdiff_t batch_w, ptrdiff_t batch_c,
                                           DecayEpilogue& ep) {
    const ptrdiff_t z = blockIdx.z;
    A += z * batch_a;
    W += z * batch_w;
    C += z * batch_c;
    if (z < ep.from) ep.rate = nullptr;
}

// How a tile's operands are loaded: element by element; vectors at a time, with bfloat16 8 or 16 bytes; 16 bytes at a time, K being whole stages (then a
// row is a 32-bit offset from the tile's first and no lane looks where K ends).
enum { SINGLE = OCT_SINGLE, HALVES = OCT_HALVES, QUADS = OCT_WHOLE, WHOLE };

// More than 16 rows: a workgroup on a tile of BM rows of A by BN rows of W, a wave on WM x WN of it, in stages of 32 k. A stage
// is asked for two stages ahead (a lane's eight elements, 32 bytes), split into its parts by the wave that asked and
// written to one of two LDS buffers, where an operand of a 16 x 16 x 32 product lies as its lanes read it: no read and no write meets a
// bank twice, and a stage costs one barrier that waits for no load.
template <class TA, class TW, class TC, bool ACCUM, int BM, int BN, int WM, int WN, int LOADS>
__global__ void __launch_bounds__(64 * (BM / WM) * (BN / WN), 2)
gemm_plain_tile_kernel(const TA* __restrict__ A, const TW* __restrict__ W, TC* __restrict__ C, int M, int N,
                       int K, int lda, int ldw, int ldc, ptrdiff_t batch_a, ptrdiff_t batch_w, ptrdiff_t batch_c,
                       DecayEpilogue ep) {
    to_product(A, W, C, batch_a, batch_w, batch_c, ep);
    constexpr int WAVES = (BM / WM) * (BN / WN), STAGE = 32, STAGES = K_BLOCK / STAGE, AHEAD = (BM + BN) / 16 / WAVES > 2 ? 2 : 4;
    constexpr int AB = BM / 16, WB = BN / 16;                            // blocks of 16 rows of a tile's operands
    constexpr bool EITHER = AB % WAVES != 0;                             // of which a wave stages one, of either operand, or so many of both
    constexpr int AU = EITHER ? 1 : AB / WAVES, WU = EITHER ? 1 : WB / WAVES;
    constexpr int MB = WM / 16, NB = WN / 16;                            // and multiplies so many
    constexpr int AP = Parts<TA>::COUNT, WP = Parts<TW>::COUNT;
    static_assert(EITHER ? AB == WB && AB + WB == WAVES && std::is_same<TA, TW>::value && LOADS == WHOLE : WB % WAVES == 0, "every wave stages whole blocks");
    typedef SplitOrder<WP, AP> order;
    __shared__ __attribute__((aligned(16))) bf16x8 a_lds[2 * AB * AP * HB_WAVE], w_lds[2 * WB * WP * HB_WAVE];   // [buffer][block][part][lane]
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 15, q = lane >> 4;
    const unsigned across = (N + BN - 1) / BN, tile = blockIdx.y * gridDim.x + blockIdx.x;   // (tiles of a row of tiles)
    if (tile / across >= (unsigned)(M + BM - 1) / BM) return;
    const int m0 = (int)(tile / across) * BM, n0 = (int)(tile % across) * BN;
    const int wm = wave % (BM / WM) * MB, wn = wave / (BM / WM) * NB;    // (in blocks)
    // rows beyond M or N are the tile's first once more, whose sums go nowhere; rows lie as far apart as they may, but where 32 bits are known to do
    typedef typename std::conditional<LOADS == WHOLE, unsigned, size_t>::type Offset;
    const TA* const a_tile = A + (size_t)m0 * lda;
    const TW* const w_tile = W + (size_t)n0 * ldw;
    Offset a_row[AU], w_row[WU];
#pragma unroll
    for (int i = 0; i < AU; ++i) {
        const int row = 16 * ((EITHER ? wave % AB : wave * AU) + i) + r;
        a_row[i] = (m0 + row < M ? row : 0) * (Offset)lda + (LOADS == WHOLE ? 8 * q : 0);
    }
#pragma unroll
    for (int i = 0; i < WU; ++i) {
        const int row = 16 * ((EITHER ? wave % WB : wave * WU) + i) + r;
        w_row[i] = (n0 + row < N ? row : 0) * (Offset)ldw + (LOADS == WHOLE ? 8 * q : 0);
    }
    const bool stages_w = EITHER && wave >= AB;
    Oct<TA> a_next[AHEAD][AU];
    Oct<TW> w_next[AHEAD][WU];
    auto fetch = [&](int s, Oct<TA>* a, Oct<TW>* w) {
        const int k = s * STAGE, from = LOADS == WHOLE && k > K - STAGE ? K - STAGE : k;      // (a stage beyond K is the last once more)
        if constexpr (EITHER) {
            a[0] = load_oct<QUADS>((stages_w ? w_tile : a_tile) + from, stages_w ? w_row[0] : a_row[0]);
            return;
        }
#pragma unroll
        for (int i = 0; i < AU; ++i)
            a[i] = LOADS == WHOLE ? load_oct<QUADS>(a_tile + from, a_row[i]) : load_oct<LOADS == WHOLE ? QUADS : LOADS>(a_tile + a_row[i], k + 8 * q, K);
#pragma unroll
        for (int i = 0; i < WU; ++i)
            w[i] = LOADS == WHOLE ? load_oct<QUADS>(w_tile + from, w_row[i]) : load_oct<LOADS == WHOLE ? QUADS : LOADS>(w_tile + w_row[i], k + 8 * q, K);
    };
    auto cut = [&](int s, Oct<TA>* a, Oct<TW>* w) {          // what lies beyond K
        const int left = K - s * STAGE;
        if (LOADS == SINGLE || left >= STAGE) return;
#pragma unroll
        for (int i = 0; i < AU; ++i) ends(a[i], left - 8 * q);
#pragma unroll
        for (int i = 0; i < (EITHER ? 0 : WU); ++i) ends(w[i], left - 8 * q);
    };
    auto stash = [&](int buf, const Oct<TA>* a, const Oct<TW>* w) {
#pragma unroll
        for (int i = 0; i < AU; ++i) {
            const Parts<TA> parts = split(a[i]);
#pragma unroll
            for (int p = 0; p < AP; ++p)
                (stages_w ? w_lds : a_lds)[((buf * AB + (EITHER ? wave % AB : wave * AU) + i) * AP + p) * HB_WAVE + lane] = parts.part[p];
        }
#pragma unroll
        for (int i = 0; i < (EITHER ? 0 : WU); ++i) {
            const Parts<TW> parts = split(w[i]);
#pragma unroll
            for (int p = 0; p < WP; ++p) w_lds[((buf * WB + wave * WU + i) * WP + p) * HB_WAVE + lane] = parts.part[p];
        }
    };

    f32x4 top[NB][MB], low[NB][MB], total[NB][MB];
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int i = 0; i < MB; ++i) total[j][i] = top[j][i] = low[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};

    // stage s, in LDS; the one AHEAD from here is asked for, the next one written to the other buffer.
    auto step = [&](int s, int at) {
        const int buf = at & 1;
        Oct<TA>* a_near = a_next[(at + 1) % AHEAD];
        Oct<TW>* w_near = w_next[(at + 1) % AHEAD];
        cut(s + 1, a_near, w_near);
        fetch(s + AHEAD, a_next[at], w_next[at]);
        bf16x8 a[MB][AP], w[NB][WP];
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int p = 0; p < AP; ++p) a[i][p] = a_lds[((buf * AB + wm + i) * AP + p) * HB_WAVE + lane];
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int p = 0; p < WP; ++p) w[j][p] = w_lds[((buf * WB + wn + j) * WP + p) * HB_WAVE + lane];
#pragma unroll
        for (int p = 0; p < SPLIT_PRODUCTS; ++p)
            if (order::there(p)) {
#pragma unroll
                for (int j = 0; j < NB; ++j)
#pragma unroll
                    for (int i = 0; i < MB; ++i) {
                        f32x4& sums = p == SPLIT_PRODUCTS - 1 ? top[j][i] : low[j][i];
                        sums = mfma_k32(w[j][order::w[p] % WP], a[i][order::a[p] % AP], sums);
                    }
            }
        stash(buf ^ 1, a_near, w_near);
        hb_workgroup_barrier();
    };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) fetch(i, a_next[i], w_next[i]);
    cut(0, a_next[0], w_next[0]);
    stash(0, a_next[0], w_next[0]);
    hb_workgroup_barrier();
    for (int s = 0; s * STAGE < K;) {
        // (AHEAD stages at a time: what lies beyond K are zeros)
        const int left = K - s * STAGE, stop = s + (left >= K_BLOCK ? STAGES : (left + AHEAD * STAGE - 1) / (AHEAD * STAGE) * AHEAD);
        for (; s < stop; s += AHEAD)
#pragma unroll
            for (int at = 0; at < AHEAD; ++at) step(s + at, at);
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                total[j][i] += top[j][i] + low[j][i];
                top[j][i] = low[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
    }

    mend_blocks<TA, TW>(rows_of(A, lda, m0 + 16 * wm, M), W, ldw, n0 + 16 * wn, N, K, K_BLOCK, total);
#pragma unroll
    for (int i = 0; i < MB; ++i) {
        const int m = m0 + 16 * (wm + i) + r;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const int n = n0 + 16 * (wn + j) + 4 * q;
            // (one to three products: a chain's roundings are no more than those of the parts' products that are left out)
            if (LOADS == SINGLE && K < 4)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) total[j][i][e] = hb_sum_in_order(A + (size_t)m * lda, W + (size_t)(n + e) * ldw, K, K_BLOCK);
            store_quad<TC, ACCUM, LOADS != SINGLE>(C, ldc, m, n, N, total[j][i], ep);
        }
    }
}

// Few rows of A (a decode step, a short prompt): a product bound by the weights' bytes and, narrow ones, by the chain of k. A
// workgroup on 16 rows of W and MB blocks of 16 rows of A, a wave on every stretch of K_BLOCK (up to WAVE_WAVES of them at a
// time): no load waits for another wave, and a wave asks for all of its stretch of W at once (16 pieces of 8 elements a lane), for A
// some pieces ahead, and splits both in registers. The stretches' sums meet in LDS, where the first wave adds them in
// their order. Short products through a narrow middle are here too, and those of heads with a matrix each: a wave on vector products, 16 columns
// and 8 rows, which they had, took at 1 | 8 | 24 rows of bfloat16 weights (2048 x 128) 3.4 | 3.8 | 4.1 us, now 2.9 | 3.0 | 3.0; (4096 x 1024)
// 13.5 | 15.9 | 19.2, now 5.1 | 5.6 | 7.7; (16 heads of 128 x 512) 7.7 | 9.1 | 10.1, now 4.3 | 4.6 | 5.0.
#define WAVE_WAVES 8
template <class TA, class TW, class TC, bool ACCUM, int MB, int NB, int AHEAD, int HOW>
__global__ void __launch_bounds__(WAVE_WAVES * HB_WAVE, AHEAD == 8 ? 4 : 2)
gemm_plain_wave_kernel(const TA* __restrict__ A, const TW* __restrict__ W, TC* __restrict__ C, int M, int N,
                       int K, int lda, int ldw, int ldc, ptrdiff_t batch_a, ptrdiff_t batch_w, ptrdiff_t batch_c,
                       DecayEpilogue ep) {
    to_product(A, W, C, batch_a, batch_w, batch_c, ep);
    constexpr int A_AHEAD = NB > 1 ? 4 : AHEAD == 16 ? 8 : 2;
    __shared__ __attribute__((aligned(16))) f32x4 sums[WAVE_WAVES][NB][MB][HB_WAVE];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const int r = lane & 15, q = lane >> 4;
    const int n0 = blockIdx.x * 16 * NB, m0 = blockIdx.y * 16 * MB;
    // (rows beyond M or N are rows at hand once more, whose sums go nowhere; pieces beyond K are zeros)
    const TW* w_row[NB];
    const TA* a_row[MB];
#pragma unroll
    for (int j = 0; j < NB; ++j) w_row[j] = W + (size_t)(n0 + 16 * j + r < N ? n0 + 16 * j + r : n0) * ldw;
#pragma unroll
    for (int i = 0; i < MB; ++i) a_row[i] = A + (size_t)(m0 + 16 * i + r < M ? m0 + 16 * i + r : m0) * lda;
    f32x4 total[NB][MB], top[NB][MB], low[NB][MB];
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int i = 0; i < MB; ++i) total[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int first = 0; first < K; first += waves * K_BLOCK) {
        const int k0 = first + wave * K_BLOCK;
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int i = 0; i < MB; ++i) top[j][i] = low[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
        sum_stretch<AHEAD, A_AHEAD, HOW>(w_row, a_row, k0, K, q, top, low);
        if (first) __syncthreads();                  // (the round before has been read)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int i = 0; i < MB; ++i) sums[wave][j][i][lane] = top[j][i] + low[j][i];
        __syncthreads();
        if (wave == 0)
            for (int b = 0; b < waves && first + b * K_BLOCK < K; ++b)
#pragma unroll
                for (int j = 0; j < NB; ++j)
#pragma unroll
                    for (int i = 0; i < MB; ++i) total[j][i] += sums[b][j][i][lane];
    }
    if (wave) return;
    mend_blocks<TA, TW>(rows_of(A, lda, m0, M), W, ldw, n0, N, K, K_BLOCK, total);
#pragma unroll
    for (int i = 0; i < MB; ++i) {
        const int m = m0 + 16 * i + r;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const int n = n0 + 16 * j + 4 * q;
            store_quad<TC, ACCUM, true>(C, ldc, m, n, N, total[j][i], ep);
        }
    }
}

// Up to 16 rows on float32 weights whose k is so short that there
// is nothing to share: no LDS and no barrier; a wave goes through the stretches one after another, the next WAVE_DEPTH pieces of 32 k of
// W and A on their way while the WAVE_DEPTH before are multiplied. A stretch that is not whole goes by in rounds of four pieces in the kernel above,
// each waited for; here the next round is on its way. A whole one it asks for at once, and k beyond 1024 gives it more waves than one.
// Microseconds at 8 rows by this kernel | the one above: 2048 x 128 3.2 | 3.3, 4096 x 256 4.3 | 4.8, 32768 x 640 21.2 | 25.2, 32768 x 768 23.6 | 26.9,
// but where the strips are few 512 x 640 6.9 | 6.5, 2048 x 768 8.4 | 7.5, 16384 x 128 5.2 | 4.7; whole stretches 32768 x 512 17.5 | 16.6, 16384 x 1024
// 16.7 | 17.0, 4096 x 2048 18.6 | 12.7, 2048 x 8192 61 | 31.
template <class TA, class TW, class TC, bool ACCUM>
__global__ void __launch_bounds__(HB_WAVE)
gemm_plain_stream_kernel(const TA* __restrict__ A, const TW* __restrict__ W, TC* __restrict__ C, int M, int N,
                         int K, int lda, int ldw, int ldc, ptrdiff_t batch_a, ptrdiff_t batch_w, ptrdiff_t batch_c,
                         DecayEpilogue ep) {
    to_product(A, W, C, batch_a, batch_w, batch_c, ep);
    constexpr int ROUND = 32 * WAVE_DEPTH;
    static_assert(K_BLOCK % ROUND == 0, "a stretch of k is whole rounds of loads");
    const int lane = threadIdx.x, r = lane & 15, q = lane >> 4;
    const int n0 = blockIdx.x * 16;
    // (rows beyond M or N are row 0 once more, whose sums go nowhere; pieces beyond K are zeros)
    const TW* w_row = W + (size_t)(n0 + r < N ? n0 + r : 0) * ldw;
    const TA* a_row = A + (size_t)(r < M ? r : 0) * lda;
    f32x4 total = {0.f, 0.f, 0.f, 0.f}, top = total, low = total;
    Oct<TW> w_next[WAVE_DEPTH];
    Oct<TA> a_next[WAVE_DEPTH];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int d = 0; d < WAVE_DEPTH; ++d) {
            w_next[d] = load_oct<QUADS>(w_row, k0 + 32 * d + 8 * q, K);
            a_next[d] = load_oct<QUADS>(a_row, k0 + 32 * d + 8 * q, K);
        }
    };
    fetch(0);
    for (int k0 = 0; k0 < K; k0 += ROUND) {
        Oct<TW> w[WAVE_DEPTH];
        Oct<TA> a[WAVE_DEPTH];
#pragma unroll
        for (int d = 0; d < WAVE_DEPTH; ++d) w[d] = w_next[d], a[d] = a_next[d];
        const bool more = k0 + ROUND < K;
        fetch(k0 + ROUND);
        if (!more)
#pragma unroll
            for (int d = 0; d < WAVE_DEPTH; ++d) {
                ends(w[d], K - k0 - 32 * d - 8 * q);
                ends(a[d], K - k0 - 32 * d - 8 * q);
            }
#pragma unroll
        for (int d = 0; d < WAVE_DEPTH; ++d) mfma_split<TW, TA>(split(w[d]), split(a[d]), top, low);
        if (!more || (k0 + ROUND) % K_BLOCK == 0) {
            total += top + low;
            top = low = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    f32x4 sums[1][1] = {{total}};
    mend_blocks<TA, TW>(rows_of(A, lda, 0, M), W, ldw, n0, N, K, K_BLOCK, sums);
    if (r < M) store_quad<TC, ACCUM, true>(C, ldc, r, n0 + 4 * q, N, sums[0][0], ep);
}

// The kernel of a product of more than 16 rows: the one with the least estimated time, in microseconds. A wave of 16 x 16 or 32 x 32
// (x 512 of k) costs what a SIMD takes for it times the waves a SIMD gets; a tile's stage of 32 k what a CU takes for it times the
// tiles a CU gets, and no less than the chain from its reads of LDS over its products and the next stage's splitting to the barrier. Both sides float32 | one of
// them bfloat16: 16 x 16 8.0 | 5.3, 32 x 32 by a wave 16.2 | 11.5, tiles of 32 x 32 0.23 | 0.18 a stage (at least 0.295 | 0.27), 64 x 64 0.48 | 0.35,
// 128 x 128 1.35 | 0.80. Measured, microseconds by 16 x 16 / 32 x 32 / tiles of 32 / 64 / 128 [the float32 matrix instructions before], float32 weights: 17 x
// 2048 x 2048 12 / 17 / 22 / 32 / 78 [22], 17 x 4096 x 2048 17 / 22 / 22 / 32 / 78 [29] (a square is estimated at 17 whatever its weights' bytes, and taken), 128 x 2048 x
// 2048 35 / 19 / 22 / 32 / 80 [23], 200 x 4096 x 2048 103 / 58 / 60 / 34 / 80 [54], 563 x 4096 x 2048 281 / 138 / 137 / 92 / 81 [114], 563 x 6144 x 2048 417 / 206 /
// 210 / 121 / 86 [155], 563 x 2048 x 3072 248 / 131 / 113 / 89 / 118 [98]; bfloat16 weights: 64 x 2048 x 2048 13 / 14 / 20 / 26 / 49 [39], 563 x 4096 x 2048 191 / 105 /
// 109 / 69 / 51 [163].
// waves: a grid of them holds the product; whole: K is whole stages, the larger tiles take nothing else; a decay's exponentials and logarithms are a tile's own tail: not 64 of them a lane.
enum { STREAM, WAVE, WAVE_RING, WAVE_SQUARE, WAVE_HALVES, TILE_SINGLE, TILE_HALVES, TILE_QUADS, TILE_32, TILE_64, TILE_128 };
static int gemm_plain_choice(int M, int N, int K, int batch, bool both, bool whole, bool decay, bool waves) {
    auto tiles = [&](int side) { return (double)((N + side - 1ll) / side * ((M + side - 1) / side) * batch); };
    auto most = [&](int side) { return (double)(((long long)tiles(side) + 255) / 256); };
    auto larger = [](double a, double b) { return a > b ? a : b; };
    const double never = 1e30, stages = (K + 127) / 128 * 4, part = K < K_BLOCK ? (double)K / K_BLOCK : 1.0;
    const double per_simd = part * ((K + K_BLOCK - 1) / K_BLOCK) / 1024.0, least = K < K_BLOCK ? 0.2 * part : 0.5;
    const struct {
        int kernel;
        double cost;
    } all[5] = {
        {WAVE, !waves ? never : 2.6 + (both ? 8.0 : 5.3) * larger(per_simd * tiles(16), least)},
        {WAVE_SQUARE, !waves ? never : both ? 5.0 + larger(16.2 * per_simd * tiles(32), 12.0 * part) : 3.5 + larger(11.5 * per_simd * tiles(32), 10.0 * part)},
        {whole ? TILE_32 : TILE_QUADS, 2.4 + stages * (both ? larger(0.295, 0.03 + 0.23 * most(32)) : larger(0.27, 0.03 + 0.18 * most(32)))},
        {TILE_64, !whole ? never : 2.4 + stages * (both ? 0.48 : 0.35) * most(64)},
        {TILE_128, !whole || decay ? never : 3.0 + stages * (both ? 1.35 : 0.80) * most(128)}};
    int best = 0;
    for (int i = 1; i < 5; ++i) best = all[i].cost < all[best].cost ? i : best;
    return all[best].kernel;
}

#define GRID_X (1 << 22)
// What the entries take: rows as ever, and tiles of 32 x 32 that GRID_X times 512 hold (2 T sums a product).
#define HB_REQUIRE_TILES(M, N)                                                                                        \
    do {                                                                                                              \
        HB_REQUIRE((M) <= 65535 * 64, "gemm: M=%d, at most 4194240 rows are taken", M);                               \
        HB_REQUIRE((((M) + 31) / 32) * (((N) + 31ll) / 32) < (1ll << 31), "gemm: %d x %d sums exceed the grid", M, N); \
    } while (0)
template <class TA, class TW, class TC, bool ACCUM>
static void launch_as(const TA* A, const TW* W, TC* C, int M, int N, int K, int lda, int ldw, int ldc,
                      hipStream_t stream, int batch, ptrdiff_t batch_a, ptrdiff_t batch_w, ptrdiff_t batch_c, DecayEpilogue ep) {
    // (16-byte loads where rows and strides allow them, or 8-byte ones of bfloat16, 16-byte stores with either: float32 rows on bfloat16 ones, 2,052
    // elements apart, 8 x 2048 x 2048 6.2 us, 512 rows 45, element by element 47 and 158)
    auto borders = [&](int ea, int ew) {
        return K % ea == 0 && K % ew == 0 && lda % ea == 0 && ldw % ew == 0 && batch_a % ea == 0 && batch_w % ew == 0 &&
               (uintptr_t)A % (ea * sizeof(TA)) == 0 && (uintptr_t)W % (ew * sizeof(TW)) == 0 &&
               (sizeof(TC) != 4 || (N % 4 == 0 && ldc % 4 == 0 && batch_c % 4 == 0 && (uintptr_t)C % 16 == 0));
    };
    const bool vec = borders(16 / sizeof(TA), 16 / sizeof(TW)), half = !vec && borders(4, 4);
    auto tiles = [&](int high, int wide) { return (long long)((N + wide - 1) / wide) * ((M + high - 1) / high) * batch; };
    // (a grid's x holds fewer than 2^32 threads, a tile has up to 512: beyond GRID_X tiles the rest lie along its y)
    auto grid = [&](int high, int wide) {
        const long long n = tiles(high, wide) / batch, x = n < GRID_X ? n : GRID_X;
        return dim3((unsigned)x, (unsigned)((n + x - 1) / x), batch);
    };
    const int stretches = (K + K_BLOCK - 1) / K_BLOCK;
#define HB_PLAIN_TILE(BM, BN, WM, WN, LOADS)                                                                          \
    gemm_plain_tile_kernel<TA, TW, TC, ACCUM, BM, BN, WM, WN, LOADS>                                                  \
        <<<grid(BM, BN), 64 * (BM / WM) * (BN / WN), 0, stream>>>(A, W, C, M, N, K, lda, ldw, ldc, batch_a, batch_w,  \
                                                                 batch_c, ep)
#define HB_PLAIN_WAVE(MB, NB, AHEAD, HOW)                                                                             \
    gemm_plain_wave_kernel<TA, TW, TC, ACCUM, MB, NB, AHEAD, HOW>                                                     \
        <<<dim3((N + 16 * NB - 1) / (16 * NB), (M + 16 * MB - 1) / (16 * MB), batch), HB_WAVE * at_once, 0, stream>>>( \
            A, W, C, M, N, K, lda, ldw, ldc, batch_a, batch_w, batch_c, ep)
    // (Both sides of STREAM stand at its kernel. WAVE_RING holds 8 pieces of W instead of 16 and so twice the waves on a CU, for products whose waves fill
    // the chip at 16 more than once; us at 8 rows by 16 | 8 pieces, the waves in brackets: bfloat16 weights 6144 x 2048 [1536] 11.3 | 13.7, 8192 x 2048 [2048] 11.8 |
    // 14.4, 11008 x 2048 [2752] 16.1 | 16.1, 32768 x 1024 [4096] 19.8 | 19.6; float32 weights 4096 x 8192 [2048] 37.5 | 37.2, 11008 x 2048 24.8 | 25.0, 32768 x
    // 1024 32.1 | 28.8, 8192 x 8192 [4096] 68.6 | 57.2.)
    const long long strips = (N + 15ll) / 16 * batch;
    const int at_once = stretches < WAVE_WAVES ? stretches : WAVE_WAVES;
    const bool waves = M <= 4096 && (N + 15ll) / 16 * HB_WAVE * at_once < 1ll << 32;     // (the strips lie along x alone)
    const int which = half                                                      ? M <= 16 && waves ? WAVE_HALVES : TILE_HALVES
                      : !vec                                                    ? TILE_SINGLE
                      : M <= 16 && waves && sizeof(TW) == 4 && K < 1024 && K > 64 && K % K_BLOCK ? STREAM
                      : M <= 16 && waves                                        ? strips * at_once > 2048 ? WAVE_RING : WAVE
                                                                                : gemm_plain_choice(M, N, K, batch, Parts<TA>::COUNT + Parts<TW>::COUNT == 6,
                                                                                                    K % 32 == 0 && lda < 1 << 23 && ldw < 1 << 23, ep.rate != nullptr, waves);
    switch (which) {
        case STREAM:
            if constexpr (sizeof(TW) == 4)
                gemm_plain_stream_kernel<TA, TW, TC, ACCUM><<<dim3((N + 15) / 16, 1, batch), HB_WAVE, 0, stream>>>(
                    A, W, C, M, N, K, lda, ldw, ldc, batch_a, batch_w, batch_c, ep);
            break;
        case WAVE: HB_PLAIN_WAVE(1, 1, 16, QUADS); break;
        case WAVE_RING: HB_PLAIN_WAVE(1, 1, 8, QUADS); break;
        case WAVE_SQUARE: HB_PLAIN_WAVE(2, 2, 4, QUADS); break;
        // (both sides float32: the borders of 8 bytes of bfloat16 are theirs of 16, and none of these two is asked for)
        case WAVE_HALVES:
            if constexpr (sizeof(TA) == 2 || sizeof(TW) == 2) HB_PLAIN_WAVE(1, 1, 16, HALVES);
            break;
        case TILE_HALVES:
            if constexpr (sizeof(TA) == 2 || sizeof(TW) == 2) HB_PLAIN_TILE(32, 32, 16, 32, HALVES);
            break;
        case TILE_SINGLE: HB_PLAIN_TILE(32, 32, 16, 32, SINGLE); break;
        case TILE_QUADS: HB_PLAIN_TILE(32, 32, 16, 32, QUADS); break;
        case TILE_32:            // (a wave stages a block of either operand, where both are of a kind: half the splitting in a stage's chain)
            if constexpr (std::is_same<TA, TW>::value) HB_PLAIN_TILE(32, 32, 16, 16, WHOLE);
            else HB_PLAIN_TILE(32, 32, 16, 32, WHOLE);
            break;
        case TILE_64:
            if constexpr (std::is_same<TA, TW>::value) HB_PLAIN_TILE(64, 64, 16, 32, WHOLE);
            else HB_PLAIN_TILE(64, 64, 32, 32, WHOLE);
            break;
        case TILE_128: HB_PLAIN_TILE(128, 128, 64, 32, WHOLE); break;
    }
#undef HB_PLAIN_WAVE
#undef HB_PLAIN_TILE
}

template <class TA, class TW, class TC>
static void launch(const void* A, const void* W, void* C, int M, int N, int K, int lda, int ldw, int ldc,
                   int accumulate, hipStream_t stream, int batch = 1, ptrdiff_t batch_a = 0, ptrdiff_t batch_w = 0,
                   ptrdiff_t batch_c = 0, DecayEpilogue ep = DecayEpilogue{nullptr, nullptr, 1, 0.f, 0}) {
    if (accumulate)
        launch_as<TA, TW, TC, true>((const TA*)A, (const TW*)W, (TC*)C, M, N, K, lda, ldw, ldc, stream, batch, batch_a,
                                    batch_w, batch_c, ep);
    else
        launch_as<TA, TW, TC, false>((const TA*)A, (const TW*)W, (TC*)C, M, N, K, lda, ldw, ldc, stream, batch, batch_a,
                                     batch_w, batch_c, ep);
}

// C[M, N] (+)= A[M, K] * W[N, K]^T with row strides lda, ldw, ldc (in elements).
extern "C" int hb_gemm_plain(const void* A, int a_dtype, const void* W, int w_dtype, void* C, int c_dtype,
                             int M, int N, int K, int lda, int ldw, int ldc, int accumulate,
                             hipStream_t stream) {
    HB_REQUIRE(M > 0 && N > 0 && K > 0, "gemm: empty problem (M=%d, N=%d, K=%d)", M, N, K);
    HB_REQUIRE(lda >= K && ldw >= K && ldc >= N, "gemm: a row stride is smaller than its row");
    HB_REQUIRE_TILES(M, N);
    const int key = a_dtype * 4 + w_dtype * 2 + c_dtype;
    switch (key) {
        case 0: launch<float, float, float>(A, W, C, M, N, K, lda, ldw, ldc, accumulate, stream); break;
        case 1: launch<float, float, bf16>(A, W, C, M, N, K, lda, ldw, ldc, accumulate, stream); break;
        case 2: launch<float, bf16, float>(A, W, C, M, N, K, lda, ldw, ldc, accumulate, stream); break;
        case 3: launch<float, bf16, bf16>(A, W, C, M, N, K, lda, ldw, ldc, accumulate, stream); break;
        case 4: launch<bf16, float, float>(A, W, C, M, N, K, lda, ldw, ldc, accumulate, stream); break;
        case 5: launch<bf16, float, bf16>(A, W, C, M, N, K, lda, ldw, ldc, accumulate, stream); break;
        case 6: launch<bf16, bf16, float>(A, W, C, M, N, K, lda, ldw, ldc, accumulate, stream); break;
        case 7: launch<bf16, bf16, bf16>(A, W, C, M, N, K, lda, ldw, ldc, accumulate, stream); break;
        default: HB_REQUIRE(false, "gemm: unknown dtypes (%d, %d, %d)", a_dtype, w_dtype, c_dtype);
    }
    HB_CHECK_LAUNCH("gemm_plain");
    return 0;
}

// The same product, which may leave decays.
// A_log [N / D] and dt_bias [N], both or neither: the sums are a decay's pre-activations, and what is stored is
// the decay a column (float32 in and out, no accumulation). A_log == dt_bias: the decay is
// sigmoid(sum + dt_bias[n])^root instead.
extern "C" int hb_gemm_plain_decay(const void* A, int a_dtype, const void* W, int w_dtype, void* C, int c_dtype,
                                   int M, int N, int K, int lda, int ldw, int ldc, int accumulate,
                                   const float* A_log, const float* dt_bias, int D, float root,
                                   hipStream_t stream) {
    HB_REQUIRE(M > 0 && N > 0 && K > 0, "gemm: empty problem (M=%d, N=%d, K=%d)", M, N, K);
    HB_REQUIRE(lda >= K && ldw >= K && ldc >= N, "gemm: a row stride is smaller than its row");
    HB_REQUIRE((A_log == nullptr) == (dt_bias == nullptr), "gemm: a decay needs its rate and its bias");
    HB_REQUIRE(!A_log || (D > 0 && N % D == 0 && c_dtype == 0 && !accumulate),
               "gemm: a decay is float32, stored and not added, %d columns in heads of %d", N, D);
    const DecayEpilogue ep{A_log, dt_bias, A_log ? D : 1, root, 0};
    if (!A_log) return hb_gemm_plain(A, a_dtype, W, w_dtype, C, c_dtype, M, N, K, lda, ldw, ldc, accumulate, stream);
    HB_REQUIRE_TILES(M, N);
    switch (a_dtype * 2 + w_dtype) {
        case 0: launch<float, float, float>(A, W, C, M, N, K, lda, ldw, ldc, 0, stream, 1, 0, 0, 0, ep); break;
        case 1: launch<float, bf16, float>(A, W, C, M, N, K, lda, ldw, ldc, 0, stream, 1, 0, 0, 0, ep); break;
        case 2: launch<bf16, float, float>(A, W, C, M, N, K, lda, ldw, ldc, 0, stream, 1, 0, 0, 0, ep); break;
        case 3: launch<bf16, bf16, float>(A, W, C, M, N, K, lda, ldw, ldc, 0, stream, 1, 0, 0, 0, ep); break;
        default: HB_REQUIRE(false, "gemm: unknown dtypes (%d, %d)", a_dtype, w_dtype);
    }
    HB_CHECK_LAUNCH("gemm_plain");
    return 0;
}

// Two such products of float32 rows with float32 sums (no decay for the first): C0 = A0 W0^T, C1 = A1 W1^T, shapes and strides alike, in
// one launch: they wait for the same rows and not for each other, and a launch is the larger part of what one takes (8 x 2048 x 128,
// bfloat16 weights: 2.9 us, the two together 3.0; 24 rows 3.0 and 3.3).
extern "C" int hb_gemm_plain_decay_pair(const float* A0, const void* W0, float* C0, const float* A1, const void* W1, float* C1,
                                        int w_dtype, int M, int N, int K, int lda, int ldw, int ldc, const float* A_log,
                                        const float* dt_bias, int D, float root, hipStream_t stream) {
    HB_REQUIRE(M > 0 && N > 0 && K > 0, "gemm: empty problem (M=%d, N=%d, K=%d)", M, N, K);
    HB_REQUIRE(lda >= K && ldw >= K && ldc >= N, "gemm: a row stride is smaller than its row");
    HB_REQUIRE((A_log == nullptr) == (dt_bias == nullptr), "gemm: a decay needs its rate and its bias");
    HB_REQUIRE(!A_log || (D > 0 && N % D == 0), "gemm: %d columns are not heads of %d", N, D);
    HB_REQUIRE(w_dtype == 0 || w_dtype == 1, "gemm: unknown dtype (%d)", w_dtype);
    HB_REQUIRE_TILES(M, N);
    const DecayEpilogue ep{A_log, dt_bias, A_log ? D : 1, root, 1};
    const ptrdiff_t w_size = w_dtype ? 2 : 4;
    const ptrdiff_t far_a = (intptr_t)A1 - (intptr_t)A0, far_w = (intptr_t)W1 - (intptr_t)W0, far_c = (intptr_t)C1 - (intptr_t)C0;
    HB_REQUIRE(far_a % 4 == 0 && far_w % w_size == 0 && far_c % 4 == 0, "gemm: operands off their elements' borders");
    if (w_dtype) launch<float, bf16, float>(A0, W0, C0, M, N, K, lda, ldw, ldc, 0, stream, 2, far_a / 4, far_w / 2, far_c / 4, ep);
    else launch<float, float, float>(A0, W0, C0, M, N, K, lda, ldw, ldc, 0, stream, 2, far_a / 4, far_w / 4, far_c / 4, ep);
    HB_CHECK_LAUNCH("gemm_plain_pair");
    return 0;
}

// A batch of such products in one launch: product b reads A + b * batch_a, W + b * batch_w and writes
// C + b * batch_c (elements). Heads that each have a matrix of their own are such a batch: the row
// strides let every head's columns lie inside rows that all heads share.
extern "C" int hb_gemm_plain_batched(const void* A, int a_dtype, const void* W, int w_dtype, void* C, int c_dtype,
                                     int M, int N, int K, int lda, int ldw, int ldc, int batch, size_t batch_a,
                                     size_t batch_w, size_t batch_c, hipStream_t stream) {
    HB_REQUIRE(M > 0 && N > 0 && K > 0 && batch > 0, "gemm: empty problem (M=%d, N=%d, K=%d, batch=%d)", M, N, K, batch);
    HB_REQUIRE(lda >= K && ldw >= K && ldc >= N, "gemm: a row stride is smaller than its row");
    HB_REQUIRE(batch <= 65535, "gemm: batch=%d exceeds the grid", batch);
    HB_REQUIRE_TILES(M, N);
    const int key = a_dtype * 4 + w_dtype * 2 + c_dtype;
#define HB_BATCHED(TA, TW, TC) launch<TA, TW, TC>(A, W, C, M, N, K, lda, ldw, ldc, 0, stream, batch, batch_a, batch_w, batch_c)
    switch (key) {
        case 0: HB_BATCHED(float, float, float); break;
        case 1: HB_BATCHED(float, float, bf16); break;
        case 2: HB_BATCHED(float, bf16, float); break;
        case 3: HB_BATCHED(float, bf16, bf16); break;
        case 4: HB_BATCHED(bf16, float, float); break;
        case 5: HB_BATCHED(bf16, float, bf16); break;
        case 6: HB_BATCHED(bf16, bf16, float); break;
        case 7: HB_BATCHED(bf16, bf16, bf16); break;
        default: HB_REQUIRE(false, "gemm: unknown dtypes (%d, %d, %d)", a_dtype, w_dtype, c_dtype);
    }
#undef HB_BATCHED
    HB_CHECK_LAUNCH("gemm_plain_batched");
    return 0;
}
