// Matrix product in float32 arithmetic for any storage types and any sizes:
//   C[m, n] (+)= sum_k A[m, k] * W[n, k]      (weights are [out, in], k contiguous)
// It is the whole matrix path of the float32 mode and the fallback of the bfloat16
// mode for shapes its own MFMA kernels refuse. Each output is summed in stretches of K_BLOCK
// elements of k: a stretch from zero over k ascending with fused multiply-adds, then the
// stretches' sums one after another. Stretches lie at fixed places, so an output's value does
// not depend on M, on the tile or kernel it falls in, or on what else is in the batch, and yet
// a product of few rows can give every stretch a wave of its own. The matrix cores' float32
// products (v_mfma_f32_16x16x4_f32) add their four k one after another with one rounding each,
// bit for bit what fmaf gives in that order (checked on 16,384 sums of mixed magnitudes),
// and every kernel here feeds them k in ascending order. (One chain over all of k, which this
// replaced, was further from 64 bits: at K = 2048 8.1e-7 of the sums' root mean square, now 4.1e-7; at K = 12288 20e-7
// and 4.2e-7.) (hb_gemm_plain_short_k is the entry for products with a short k: it sends up to 32 float32 rows times bfloat16 rows to gemm_few_rows_kernel, whose four partial
// sums a column differ from that order by float32 rounding, and everything else here.)
// In xigh/herbert-rs: crates/backends/backend_bf16/src/kernels.rs:154-164 (float32 sums over k ascending of
// x[m, k] * float(w[n, k]), no bias); crates/backends/backend_vulkan/shaders/bf16_matmul.comp:31-60.
#include "common.h"
#include "mfma_f32.h"

HB_MODULE_ERROR_SLOT()

// Elements of k that are summed as one chain; a multiple of every kernel's stage.
#define K_BLOCK 512

// What a product may do to a sum before it stores it: nothing (rate null), or turn the pre-activation of a
// decay into the decay itself, exp(-exp(rate[n / D]) * softplus(sum + bias[n])) for column n (float32; the
// arithmetic of hb_channel_decay, which does the same to rows that lie in memory). A decay of the other kind
// (rate == bias, the mark of it): sigmoid(sum + bias[n])^root = exp(-root * softplus(-(sum + bias[n]))).
struct DecayEpilogue {
    const float* rate;
    const float* bias;
    int D;
    float root;
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

// More than 16 rows: a workgroup of four waves (2 x 2) on a tile of BM rows of A by BN rows of W. Stages of BK elements
// of k go through LDS in two buffers: a stage is asked for (16 bytes a lane) before the one at hand is multiplied and
// written to the other buffer after it, so a stage costs one barrier and no wait for memory. A product of 16 x 16 x 4
// wants k = k0 + lane / 16 from a lane, so within every 16 k LDS holds a row's elements transposed, element 4 s + q at
// place 4 q + s: a lane's next four products are then one 16-byte read. Rows are BK + 4 floats apart: the reads of 16
// rows meet no bank twice. Bound by the matrix cores (a library's large product reaches 154 TFLOP/s here):
// 4096 x 4096 x 4096 in 1,098 us (125 TFLOP/s), 564 x 6144 x 2048 in 156, 564 x 2048 x 2048 in 68, 64 x 4096 x 4096 in
// 55; the kernel of vector FMAs and 4-byte loads that this replaced took 2,465, 372, 323 and 632.
template <class TA, class TW, class TC, bool ACCUM, int BM, int BN, int BK, bool VEC>
__global__ void __launch_bounds__(256, 2)
gemm_plain_tile_kernel(const TA* __restrict__ A, const TW* __restrict__ W, TC* __restrict__ C, int M, int N,
                       int K, int lda, int ldw, int ldc, size_t batch_a, size_t batch_w, size_t batch_c,
                       DecayEpilogue ep) {
    // (blockIdx.z: one of a batch of products whose operands lie batch_* elements apart)
    A += blockIdx.z * batch_a;
    W += blockIdx.z * batch_w;
    C += blockIdx.z * batch_c;
    constexpr int LD = BK + 4, QUADS = BK / 4;
    constexpr int QA = BM * QUADS / 256, QW = BN * QUADS / 256;      // quads a thread stages of either operand
    constexpr int MB = BM / 32, NB = BN / 32;                        // blocks of 16 a wave
    __shared__ __attribute__((aligned(16))) float As[2][BM * LD], Ws[2][BN * LD];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 15, q = lane >> 4;
    const unsigned across = (N + BN - 1) / BN, tile = blockIdx.y * gridDim.x + blockIdx.x;   // (tiles of a row of tiles)
    if (tile / across >= (unsigned)(M + BM - 1) / BM) return;
    const int m0 = (int)(tile / across) * BM, n0 = (int)(tile % across) * BN;
    const int wm = (wave & 1) * (BM / 2), wn = (wave >> 1) * (BN / 2);

    f32x4 a_next[QA], w_next[QW];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < QA; ++i) {
            const int row = (tid + 256 * i) / QUADS, k = k0 + 4 * ((tid + 256 * i) % QUADS);
            a_next[i] = load_quad<VEC>(A + (size_t)(m0 + row) * lda + k, m0 + row < M ? K - k : 0);
        }
#pragma unroll
        for (int i = 0; i < QW; ++i) {
            const int row = (tid + 256 * i) / QUADS, k = k0 + 4 * ((tid + 256 * i) % QUADS);
            w_next[i] = load_quad<VEC>(W + (size_t)(n0 + row) * ldw + k, n0 + row < N ? K - k : 0);
        }
    };
    auto stash = [&](int buf) {
#pragma unroll
        for (int i = 0; i < QA; ++i) {
            const int row = (tid + 256 * i) / QUADS, quad = (tid + 256 * i) % QUADS;
            float* to = &As[buf][row * LD + (quad & ~3) * 4 + (quad & 3)];
            to[0] = a_next[i][0], to[4] = a_next[i][1], to[8] = a_next[i][2], to[12] = a_next[i][3];
        }
#pragma unroll
        for (int i = 0; i < QW; ++i) {
            const int row = (tid + 256 * i) / QUADS, quad = (tid + 256 * i) % QUADS;
            float* to = &Ws[buf][row * LD + (quad & ~3) * 4 + (quad & 3)];
            to[0] = w_next[i][0], to[4] = w_next[i][1], to[8] = w_next[i][2], to[12] = w_next[i][3];
        }
    };

    static_assert(K_BLOCK % BK == 0, "a stretch of k is whole stages");
    f32x4 acc[NB][MB], total[NB][MB];
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int i = 0; i < MB; ++i) total[j][i] = acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};

    fetch(0);
    stash(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += BK, buf ^= 1) {
        const bool more = k0 + BK < K;
        if (more) fetch(k0 + BK);
#pragma unroll
        for (int b = 0; b < BK / 16; ++b) {
            f32x4 a[MB], w[NB];
#pragma unroll
            for (int i = 0; i < MB; ++i) a[i] = *(const f32x4*)&As[buf][(wm + 16 * i + r) * LD + 16 * b + 4 * q];
#pragma unroll
            for (int j = 0; j < NB; ++j) w[j] = *(const f32x4*)&Ws[buf][(wn + 16 * j + r) * LD + 16 * b + 4 * q];
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int j = 0; j < NB; ++j)
#pragma unroll
                    for (int i = 0; i < MB; ++i) acc[j][i] = mfma_k4(w[j][s], a[i][s], acc[j][i]);
        }
        if (more) stash(buf ^ 1);
        if (!more || (k0 + BK) % K_BLOCK == 0) {
#pragma unroll
            for (int j = 0; j < NB; ++j)
#pragma unroll
                for (int i = 0; i < MB; ++i) total[j][i] += acc[j][i], acc[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        __syncthreads();
    }

#pragma unroll
    for (int i = 0; i < MB; ++i) {
        const int m = m0 + wm + 16 * i + r;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < NB; ++j)
            store_quad<TC, ACCUM, VEC>(C, ldc, m, n0 + wn + 16 * j + 4 * q, N, total[j][i], ep);
    }
}

// Up to 16 rows (a decode step): a product bound by the weights' bytes and, narrow ones, by the chain of k. A workgroup
// on 16 rows of W, a wave on every stretch of K_BLOCK (up to WAVE_WAVES of them at a time): no load waits for another
// wave, and a wave asks for all of its stretch of W at once (32 quads a lane), for A eight blocks of 16 k ahead; the
// lanes' quads are transposed in registers. The stretches' sums meet in LDS, where a thread an output adds them in
// their order. 2 x 2048 x 2048 takes 10.7 us (one wave for all of k, a chain of 512 products with eight blocks in
// flight: 19.4), 2 x 2048 x 3072 12.8 (27.9), 2 x 4096 x 2048 13.3 (20.0), 8 x 4096 x 12288 62 (106); with bfloat16
// weights 10.5 (36), 12.9 (53), 11 (38) and 43 (233).
#define WAVE_ROWS 16
#define WAVE_WAVES 8
#define WAVE_DEPTH 8
template <class TA, class TW, class TC, bool ACCUM>
__global__ void __launch_bounds__(WAVE_WAVES * HB_WAVE)
gemm_plain_wave_kernel(const TA* __restrict__ A, const TW* __restrict__ W, TC* __restrict__ C, int M, int N,
                       int K, int lda, int ldw, int ldc, size_t batch_a, size_t batch_w, size_t batch_c,
                       DecayEpilogue ep) {
    A += blockIdx.z * batch_a;
    W += blockIdx.z * batch_w;
    C += blockIdx.z * batch_c;
    constexpr int GROUPS = K_BLOCK / 16 / WAVE_DEPTH;
    __shared__ __attribute__((aligned(16))) f32x4 sums[WAVE_WAVES][HB_WAVE];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const int r = lane & 15, q = lane >> 4;
    const int n0 = blockIdx.x * 16;
    // (rows beyond M or N are row 0 once more, whose sums go nowhere; blocks beyond K are zeros)
    const TW* w_row = W + (size_t)(n0 + r < N ? n0 + r : 0) * ldw + 4 * q;
    const TA* a_row = A + (size_t)(r < M ? r : 0) * lda + 4 * q;
    f32x4 total = {0.f, 0.f, 0.f, 0.f};
    for (int first = 0; first < K; first += waves * K_BLOCK) {
        const int k0 = first + wave * K_BLOCK;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        if (k0 + K_BLOCK <= K) {
            f32x4 w[GROUPS][WAVE_DEPTH], a[2][WAVE_DEPTH];
            auto fetch_a = [&](int g) {
#pragma unroll
                for (int d = 0; d < WAVE_DEPTH; ++d) a[g & 1][d] = load_quad<true>(a_row + k0 + 16 * (g * WAVE_DEPTH + d), 4);
            };
            fetch_a(0);
#pragma unroll
            for (int g = 0; g < GROUPS; ++g)
#pragma unroll
                for (int d = 0; d < WAVE_DEPTH; ++d) w[g][d] = load_quad<true>(w_row + k0 + 16 * (g * WAVE_DEPTH + d), 4);
#pragma unroll
            for (int g = 0; g < GROUPS; ++g) {
                if (g + 1 < GROUPS) fetch_a(g + 1);
#pragma unroll
                for (int d = 0; d < WAVE_DEPTH; ++d) {
                    transpose_quads(w[g][d]);
                    transpose_quads(a[g & 1][d]);
#pragma unroll
                    for (int s = 0; s < 4; ++s) acc = mfma_k4(w[g][d][s], a[g & 1][d][s], acc);
                }
            }
        } else {
            for (int k = k0; k < K; k += 16) {       // (what is left of k, blocks of 16)
                f32x4 w = load_quad<true>(w_row + k, 4), a = load_quad<true>(a_row + k, 4);
                transpose_quads(w);
                transpose_quads(a);
#pragma unroll
                for (int s = 0; s < 4; ++s) acc = mfma_k4(w[s], a[s], acc);
            }
        }
        if (first) __syncthreads();                  // (the round before has been read)
        sums[wave][lane] = acc;
        __syncthreads();
        if (wave == 0)
            for (int b = 0; b < waves && first + b * K_BLOCK < K; ++b) total += sums[b][lane];
    }
    if (wave == 0 && r < M) store_quad<TC, ACCUM, true>(C, ldc, r, n0 + 4 * q, N, total, ep);
}

// The same rows for float32 weights that fill the chip with a wave for every 16 of their rows, or whose k is so short that there
// is nothing to share: no LDS and no barrier; a wave goes through the stretches one after another, the next WAVE_DEPTH blocks of 16 k of
// W and A on their way while the WAVE_DEPTH before are multiplied. Microseconds by the kernel above / this one, two rows: 4096 x 480 10.8 /
// 6.8, 2048 x 896 10.8 / 10.0, 4096 x 1024 9.4 / 11.3, 8192 x 1024 13.8 / 12.5, 8192 x 1504 20.7 / 17.3, 8192 x 2048 20.1 / 21.7, 12288 x 2048 24.1 /
// 23.6, 12288 x 4096 46.7 / 42.2, 32768 x 2048 61.6 / 54.6, 4096 x 64 2.9 / 3.0, 4096 x 16 2.4 / 3.1. With bfloat16 weights it is the slower one
// everywhere (32768 x 2048 46.9 / 79.4).
template <class TA, class TW, class TC, bool ACCUM>
__global__ void __launch_bounds__(HB_WAVE)
gemm_plain_stream_kernel(const TA* __restrict__ A, const TW* __restrict__ W, TC* __restrict__ C, int M, int N,
                         int K, int lda, int ldw, int ldc, size_t batch_a, size_t batch_w, size_t batch_c,
                         DecayEpilogue ep) {
    A += blockIdx.z * batch_a;
    W += blockIdx.z * batch_w;
    C += blockIdx.z * batch_c;
    static_assert(K_BLOCK % (16 * WAVE_DEPTH) == 0, "a stretch of k is whole rounds of loads");
    const int lane = threadIdx.x, r = lane & 15, q = lane >> 4;
    const int n0 = blockIdx.x * 16;
    // (rows beyond M or N are row 0 once more, whose sums go nowhere; blocks beyond K are zeros)
    const TW* w_row = W + (size_t)(n0 + r < N ? n0 + r : 0) * ldw + 4 * q;
    const TA* a_row = A + (size_t)(r < M ? r : 0) * lda + 4 * q;
    f32x4 total = {0.f, 0.f, 0.f, 0.f}, acc = total, w_next[WAVE_DEPTH], a_next[WAVE_DEPTH];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int d = 0; d < WAVE_DEPTH; ++d) {
            const int k = k0 + 16 * d;
            w_next[d] = load_quad<true>(w_row + k, K - k);
            a_next[d] = load_quad<true>(a_row + k, K - k);
        }
    };
    fetch(0);
    for (int k0 = 0; k0 < K; k0 += 16 * WAVE_DEPTH) {
        f32x4 w[WAVE_DEPTH], a[WAVE_DEPTH];
#pragma unroll
        for (int d = 0; d < WAVE_DEPTH; ++d) w[d] = w_next[d], a[d] = a_next[d];
        const bool more = k0 + 16 * WAVE_DEPTH < K;
        if (more) fetch(k0 + 16 * WAVE_DEPTH);
#pragma unroll
        for (int d = 0; d < WAVE_DEPTH; ++d) {
            transpose_quads(w[d]);
            transpose_quads(a[d]);
#pragma unroll
            for (int s = 0; s < 4; ++s) acc = mfma_k4(w[d][s], a[d][s], acc);
        }
        if (!more || (k0 + 16 * WAVE_DEPTH) % K_BLOCK == 0) total += acc, acc = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    if (r < M) store_quad<TC, ACCUM, true>(C, ldc, r, n0 + 4 * q, N, total, ep);
}

// The kernel of a product. 16-byte loads and stores where rows and strides allow them. Up to 16 rows of whole blocks of
// 16 k take one of the two kernels above. Beyond, the tile with the least estimated time: what a CU spends on one (microseconds at K = 2048 on all
// CUs: 128 x 128 137, alone on a CU 152; 64 x 64 43.5 and 52; 32 x 32 12.8, of which four or more share a CU and few are left over) times
// the most that a CU gets. Measured by 128 / 64 / 32: 564 x 6144 x 2048 156 / 168 / 173 us, 564 x 4096 x 2048 155 / 132 / 116, 564 x 2048 x
// 2048 152 / 87 / 68, 1200 x 4096 x 4096 546 / 419 / 456, 4096 x 4096 x 4096 1,098 / 1,307 / 1,489. (Tiles of 64 x 32: 162, 115, 72.)
#define GRID_X (1 << 23)
// What the entries take: rows as ever, and tiles of 32 x 32 that GRID_X times 256 hold (2 T sums a product).
#define HB_REQUIRE_TILES(M, N)                                                                                        \
    do {                                                                                                              \
        HB_REQUIRE((M) <= 65535 * 64, "gemm: M=%d, at most 4194240 rows are taken", M);                               \
        HB_REQUIRE((((M) + 31) / 32) * (((N) + 31ll) / 32) < (1ll << 31), "gemm: %d x %d sums exceed the grid", M, N); \
    } while (0)
template <class TA, class TW, class TC, bool ACCUM>
static void launch_as(const TA* A, const TW* W, TC* C, int M, int N, int K, int lda, int ldw, int ldc,
                      hipStream_t stream, int batch, size_t batch_a, size_t batch_w, size_t batch_c, DecayEpilogue ep) {
    const bool vec = K % 4 == 0 && lda % 4 == 0 && ldw % 4 == 0 && batch_a % 4 == 0 && batch_w % 4 == 0 &&
                     (uintptr_t)A % (4 * sizeof(TA)) == 0 && (uintptr_t)W % (4 * sizeof(TW)) == 0 &&
                     (sizeof(TC) != 4 || (N % 4 == 0 && ldc % 4 == 0 && batch_c % 4 == 0 && (uintptr_t)C % 16 == 0));
    auto tiles = [&](int side) { return (long long)((N + side - 1) / side) * ((M + side - 1) / side) * batch; };
    // (a grid's x holds fewer than 2^32 threads: beyond GRID_X tiles the rest lie along its y)
    auto grid = [&](int side) {
        const long long n = tiles(side) / batch, x = n < GRID_X ? n : GRID_X;
        return dim3((unsigned)x, (unsigned)((n + x - 1) / x), batch);
    };
    const int stretches = (K + K_BLOCK - 1) / K_BLOCK, wave_threads = HB_WAVE * (stretches < WAVE_WAVES ? stretches : WAVE_WAVES);
    auto most = [&](int side) { return (double)((tiles(side) + 255) / 256); };
    // (a decay's exponentials and logarithms are a tile's own tail: not 64 of them a lane)
    const double large = ep.rate ? 1e30 : tiles(128) <= 256 ? 152.0 : 137.0 * most(128), medium = tiles(64) <= 256 ? 52.0 : 43.5 * most(64),
                 small = 12.8 * (tiles(32) <= 460 ? 1.8 : tiles(32) / 256.0);
#define HB_PLAIN_TILE(BM, BK, VEC)                                                                                    \
    gemm_plain_tile_kernel<TA, TW, TC, ACCUM, BM, BM, BK, VEC>                                                        \
        <<<grid(BM), 256, 0, stream>>>(A, W, C, M, N, K, lda, ldw, ldc, batch_a, batch_w, batch_c, ep)
    // (both sides of these lines stand at gemm_plain_stream_kernel)
    const long long strips = (N + 15ll) / 16 * batch;
    const bool streams = sizeof(TW) == 4 && K > 64 && (K < 1024 || strips >= 768 || (K < 2048 && strips >= 512));
    if (vec && M <= WAVE_ROWS && K % 16 == 0 && streams) {
        if constexpr (sizeof(TW) == 4)
            gemm_plain_stream_kernel<TA, TW, TC, ACCUM><<<dim3((N + 15) / 16, 1, batch), HB_WAVE, 0, stream>>>(
                A, W, C, M, N, K, lda, ldw, ldc, batch_a, batch_w, batch_c, ep);
    }
    else if (vec && M <= WAVE_ROWS && K % 16 == 0)
        gemm_plain_wave_kernel<TA, TW, TC, ACCUM><<<dim3((N + 15) / 16, 1, batch), wave_threads, 0, stream>>>(
            A, W, C, M, N, K, lda, ldw, ldc, batch_a, batch_w, batch_c, ep);
    else if (!vec)
        HB_PLAIN_TILE(32, 64, false);
    else if (large <= medium && large <= small)
        HB_PLAIN_TILE(128, 32, true);
    else if (medium <= small)
        HB_PLAIN_TILE(64, 64, true);
    else
        HB_PLAIN_TILE(32, 64, true);
#undef HB_PLAIN_TILE
}

template <class TA, class TW, class TC>
static void launch(const void* A, const void* W, void* C, int M, int N, int K, int lda, int ldw, int ldc,
                   int accumulate, hipStream_t stream, int batch = 1, size_t batch_a = 0, size_t batch_w = 0,
                   size_t batch_c = 0, DecayEpilogue ep = DecayEpilogue{nullptr, nullptr, 1, 0.f}) {
    if (accumulate)
        launch_as<TA, TW, TC, true>((const TA*)A, (const TW*)W, (TC*)C, M, N, K, lda, ldw, ldc, stream, batch, batch_a,
                                    batch_w, batch_c, ep);
    else
        launch_as<TA, TW, TC, false>((const TA*)A, (const TW*)W, (TC*)C, M, N, K, lda, ldw, ldc, stream, batch, batch_a,
                                     batch_w, batch_c, ep);
}


// Few rows times a matrix of bfloat16 rows with a short k (the second product of a pair through a narrow
// middle, one token a sequence). Bound by latency: the wave kernel above is one chain of all of k. Here a wave takes
// 16 output columns, four lanes a column, each lane a quarter of k in steps of 8
// (one 16-byte load of the weights' row), for up to 8 rows of A at once, which the wave first copies to
// LDS so that no load waits for another; the four partial sums meet by two lane exchanges. Float32
// arithmetic throughout. A's rows and W's rows must be 16-byte aligned, K in steps of 32 up to FEW_ROWS_K.
// Microseconds, beside gemm_plain's kernel for the same rows (up to 16 the wave kernel, beyond tiles of 32 x 32):
//   N x K          1 row          8             16            24            32
//   2048 x 128     3.4 / 3.7      3.7 / 3.8     3.8 / 3.9     4.0 / 3.7     4.1 / 3.9
//   4096 x 256     4.9 / 5.5      5.6 / 5.6     6.4 / 5.7     6.8 / 5.8     7.8 / 5.8
//   4096 x 1024    14.8 / 19.4    17.0 / 19.4   18.9 / 19.5   19.8 / 20.8   23.3 / 20.9
// It pays up to 8 rows and, where k is long, up to 24; the line at 32 rows (few_rows_takes) is older than the two others.
#define FEW_ROWS_M 8
#define FEW_ROWS_K 1024
__global__ void __launch_bounds__(HB_WAVE)
gemm_few_rows_kernel(const float* __restrict__ A, const bf16* __restrict__ W, float* __restrict__ C, int M, int N,
                     int K, int lda, int ldw, int ldc, DecayEpilogue ep, size_t batch_a = 0, size_t batch_w = 0,
                     size_t batch_c = 0) {
    // (blockIdx.z: one of a batch of products whose operands lie batch_* elements apart)
    A += blockIdx.z * batch_a;
    W += blockIdx.z * batch_w;
    C += blockIdx.z * batch_c;
    __shared__ __attribute__((aligned(16))) float rows_of_a[FEW_ROWS_M * FEW_ROWS_K];
    const int lane = threadIdx.x;
    const int n = blockIdx.x * 16 + lane / 4;
    const int part = lane % 4;
    const int m0 = blockIdx.y * FEW_ROWS_M;
    const int rows = M - m0 < FEW_ROWS_M ? M - m0 : FEW_ROWS_M;
    const int quarter = K / 4;
    for (int idx = lane; idx < FEW_ROWS_M * quarter; idx += HB_WAVE) {
        const int i = idx / quarter, f = idx % quarter;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (i < rows) v = *(const float4*)(A + (size_t)(m0 + i) * lda + 4 * f);
        *(float4*)&rows_of_a[i * K + 4 * f] = v;
    }
    __syncthreads();
    float acc[FEW_ROWS_M];
#pragma unroll
    for (int i = 0; i < FEW_ROWS_M; ++i) acc[i] = 0.f;
    if (n < N) {
        const bf16* w_row = W + (size_t)n * ldw + part * quarter;
        const float* a_row = rows_of_a + part * quarter;
        for (int k = 0; k < quarter; k += 8) {
            const uint4 packed = *(const uint4*)(w_row + k);
            float w[8];
            w[0] = __uint_as_float(packed.x << 16), w[1] = __uint_as_float(packed.x & 0xffff0000u);
            w[2] = __uint_as_float(packed.y << 16), w[3] = __uint_as_float(packed.y & 0xffff0000u);
            w[4] = __uint_as_float(packed.z << 16), w[5] = __uint_as_float(packed.z & 0xffff0000u);
            w[6] = __uint_as_float(packed.w << 16), w[7] = __uint_as_float(packed.w & 0xffff0000u);
#pragma unroll
            for (int i = 0; i < FEW_ROWS_M; ++i) {
                const float4 lo = *(const float4*)(a_row + i * K + k);
                const float4 hi = *(const float4*)(a_row + i * K + k + 4);
                float s = acc[i];
                s = fmaf(lo.x, w[0], s), s = fmaf(lo.y, w[1], s), s = fmaf(lo.z, w[2], s), s = fmaf(lo.w, w[3], s);
                s = fmaf(hi.x, w[4], s), s = fmaf(hi.y, w[5], s), s = fmaf(hi.z, w[6], s), s = fmaf(hi.w, w[7], s);
                acc[i] = s;
            }
        }
    }
#pragma unroll
    for (int i = 0; i < FEW_ROWS_M; ++i) {
        acc[i] += __shfl_xor(acc[i], 1, HB_WAVE);
        acc[i] += __shfl_xor(acc[i], 2, HB_WAVE);
    }
    // (all four lanes of a column hold its sums: each stores, and first turns into a decay, every fourth row)
    static_assert(FEW_ROWS_M % 4 == 0, "the rows are dealt out to a column's four lanes");
#pragma unroll
    for (int j = 0; j < FEW_ROWS_M / 4; ++j) {
        const float s = part == 0 ? acc[4 * j] : part == 1 ? acc[4 * j + 1] : part == 2 ? acc[4 * j + 2] : acc[4 * j + 3];
        const int i = 4 * j + part;
        if (n < N && i < rows) C[(size_t)(m0 + i) * ldc + n] = ep.rate ? decay_of(ep, s, n) : s;
    }
}

static bool few_rows_takes(const void* A, int a_dtype, const void* W, int w_dtype, int c_dtype, int M, int K, int lda,
                           int ldw, int accumulate) {
    return a_dtype == 0 && w_dtype == 1 && c_dtype == 0 && !accumulate && M <= 32 && K % 32 == 0 && K <= FEW_ROWS_K && lda % 4 == 0 &&
           ldw % 8 == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0;
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

// The same product for callers whose k is short (a narrow middle): few rows take the kernel made for them.
// A_log [N / D] and dt_bias [N], both or neither: the sums are a decay's pre-activations, and what is stored is
// the decay a column (float32 in and out, no accumulation). A_log == dt_bias: the decay is
// sigmoid(sum + dt_bias[n])^root instead.
extern "C" int hb_gemm_plain_short_k(const void* A, int a_dtype, const void* W, int w_dtype, void* C, int c_dtype,
                                     int M, int N, int K, int lda, int ldw, int ldc, int accumulate,
                                     const float* A_log, const float* dt_bias, int D, float root,
                                     hipStream_t stream) {
    HB_REQUIRE(M > 0 && N > 0 && K > 0, "gemm: empty problem (M=%d, N=%d, K=%d)", M, N, K);
    HB_REQUIRE(lda >= K && ldw >= K && ldc >= N, "gemm: a row stride is smaller than its row");
    HB_REQUIRE((A_log == nullptr) == (dt_bias == nullptr), "gemm: a decay needs its rate and its bias");
    HB_REQUIRE(!A_log || (D > 0 && N % D == 0 && c_dtype == 0 && !accumulate),
               "gemm: a decay is float32, stored and not added, %d columns in heads of %d", N, D);
    const DecayEpilogue ep{A_log, dt_bias, A_log ? D : 1, root};
    if (few_rows_takes(A, a_dtype, W, w_dtype, c_dtype, M, K, lda, ldw, accumulate)) {
        gemm_few_rows_kernel<<<dim3((N + 15) / 16, (M + FEW_ROWS_M - 1) / FEW_ROWS_M), HB_WAVE, 0, stream>>>(
            (const float*)A, (const bf16*)W, (float*)C, M, N, K, lda, ldw, ldc, ep);
        HB_CHECK_LAUNCH("gemm_few_rows");
        return 0;
    }
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
    // few rows (one token a sequence) with a short k: the kernel made for them, a product of the batch a grid's layer
    if (few_rows_takes(A, a_dtype, W, w_dtype, c_dtype, M, K, lda, ldw, 0) && batch_a % 4 == 0 && batch_w % 8 == 0) {
        gemm_few_rows_kernel<<<dim3((N + 15) / 16, (M + FEW_ROWS_M - 1) / FEW_ROWS_M, batch), HB_WAVE, 0, stream>>>(
            (const float*)A, (const bf16*)W, (float*)C, M, N, K, lda, ldw, ldc, DecayEpilogue{nullptr, nullptr, 1, 0.f},
            batch_a, batch_w, batch_c);
        HB_CHECK_LAUNCH("gemm_few_rows_batched");
        return 0;
    }
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
