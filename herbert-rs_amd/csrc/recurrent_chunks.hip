// The gated delta rule and the linear attention with a decay a key channel (recurrent.hip has the rules and the walk
// token by token) for portions of many tokens: 64 tokens of a head at a time as float32 products on the matrix cores.
// The walk is a chain of tokens, 0.38 us each whatever the GPU has free; here the chain is one of chunks.
//
// Within a chunk, with G_t the product of the decays up to token t (a vector over the key's entries), S_0 the state before it:
//   u_t = beta_t (v_t - S_0^T (G_t k_t) - sum_(i<t) A_ti u_i),    A_ti = sum_d k_t k_i G_t / G_i
//   o_t = S_0^T (G_t q_t) + sum_(i<=t) B_ti u_i,                  B_ti = sum_d q_t k_i G_t / G_i
//   S   = G_64 S_0 + sum_i (G_64 / G_i k_i) u_i^T
// so U = T (beta V) - T (beta G K) S_0 with T = (I + beta A)^-1, unit lower triangular. (The linear attention has u = v.)
// No quotient of decays is ever formed: G_t / G_i is a product of the decays between, which can go to zero but not
// beyond one. For pairs of tokens in different blocks of 16 it is split where the later block begins. Within a block
// the pairs are taken in four levels, s = 1, 2, 4, 8: pairs whose halves of a run of 2 s tokens differ, split in the
// middle of that run; the products over runs grow from level to level by one exchange between the lanes of 16 tokens.
//
// This is the chunked form of the delta rule with gates by Yang, Kautz and Hatamizadeh (Gated Delta Networks, 2024; without
// gates Yang, Wang, Zhang, Shen and Kim, 2024) and of gated linear attention (Yang, Wang, Shen, Panda and Kim, 2023); T is
// the triangular factor of a product of Householder-like matrices (Bischof and Van Loan, 1987). The levels are this file's.
//
// chunk_prepare_kernel: everything that does not need S_0, one workgroup a (chunk, head), all of them at once. It leaves
// in scratch, as the operands that the second kernel's lanes load: G q, G_64 / G k, B, and -T beta G K and T beta V.
// chunk_scan_kernel: the chain of chunks, one workgroup a (head, 16 columns of S): four waves for the chain, each 16 tokens of a
// chunk (U) and a quarter of the state's rows (S), and four for the outputs (O), 16 tokens each.
//
// The walk rounds the state and what is subtracted from a value token by token; here a rounding of A, B or T reaches
// many tokens. So A, B and T are sums in float64 (the decays of the delta rule too), rounded once; sums over tokens run in their order, the
// latest and mostly largest last; sums over a key's entries are eight chains of float32 added in pairs. Against 64 bits, 333 tokens, 16
// heads of 64 or 128, keys of unit length drawn at random or with cosines of 0.5 or 0.8, decays spread over (0, 1) or around 0.5 to
// 0.999: the outputs' error is 0.67 to 0.97 of the walk's (0.8e-7 to 1e-6), 0.56 to 0.88 for the linear attention, and that of the
// state left 0.76 to 1.06. (With A, B and T in float32 the outputs' was up to 1.3 of the walk's, the state's up to 2.)
//
// 2,048 tokens of 16 heads of 128 x 128 take 141 us (the walk 781), with a decay a channel 199 (1,084), the linear attention
// 131 (909); 8 sequences of 300 tokens with a decay a channel 217 (408), the linear attention 123 (455). Bound: the second kernel by its
// chain (64 products of 32 cycles a chunk and wave and two exchanges through LDS, 100 us of the 141), the first by its products in
// float64 of 64 cycles and what lies between them. With one decay a head its pairs within a block are summed once instead of once a
// level (256 of 448 products of its longest wave), and its pieces lie in LDS twice over, so that two workgroups fit a CU: 86 us -> 52, though
// half of the registers are 27 too few for keys of 128 (112 bytes a lane in memory). With a decay a channel and keys of 64 two are 25 too few
// and still ahead, both kernels: 2,048 tokens of 16 heads 116 us -> 105, four times that of 32 heads 596 -> 477, 128 tokens 32.4 -> 33.4. With
// keys of 128 a lane's decays take more than half of the registers: one workgroup a CU (two spill 270 of them).
#include "common.h"
#include "mfma_f32.h"
#include <math.h>
#include <type_traits>

HB_MODULE_ERROR_SLOT()

#define CHUNK 64

// Where a (chunk, head)'s pieces lie in its part of the scratch, in floats.
struct ChunkLayout {
    int q, k, b, w, u, g, from, lost, size;
};
__host__ __device__ inline ChunkLayout chunk_layout(int D, int V, bool delta) {
    ChunkLayout l;
    l.q = 0;                              // [4 blocks of tokens][D / 16][64 lanes][4]: G q, rows of tokens
    l.k = l.q + CHUNK * D;                // [D / 16][4][64][4]: G_64 / G k, rows of key entries
    l.b = l.k + CHUNK * D;                // [4][4][64][4]: B, rows of tokens
    l.w = l.b + CHUNK * CHUNK;            // [4][D / 16][64][4]: -T beta G K, rows of tokens
    l.u = l.w + (delta ? CHUNK * D : 0);  // [4][V / 16][64][4]: T beta V, as sums lie
    l.g = l.u + (delta ? CHUNK * V : 0);  // [D]: G_64
    l.from = l.g + D;                     // [V] int: the token from which a column is not finite (64: none)
    l.lost = l.from + V;                  // [4] int: a bit for each of a block's tokens whose query is not finite
    l.size = l.lost + 4;
    return l;
}

__device__ __forceinline__ int in_quads(int i) { return (i & ~15) + 4 * (i & 3) + ((i >> 2) & 3); }
// A sum over a key's entries as N chains that are added in pairs, as the walk adds its lanes' sums.
template <int N>
struct Chains {
    f32x4 part[N];
    __device__ __forceinline__ Chains() {
#pragma unroll
        for (int i = 0; i < N; ++i) part[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    __device__ __forceinline__ void add(float w, float a, int i) { part[i % N] = mfma_k4(w, a, part[i % N]); }
    __device__ __forceinline__ f32x4 sum() const {
        f32x4 t[N];
#pragma unroll
        for (int i = 0; i < N; ++i) t[i] = part[i];
#pragma unroll
        for (int n = N / 2; n > 0; n /= 2)
#pragma unroll
            for (int i = 0; i < n; ++i) t[i] += t[i + n];
        return t[0];
    }
};
typedef double f64x4 __attribute__((ext_vector_type(4)));
// mfma_k4 in float64; lane l's four sums are those of n = 4 e + l / 16 (not 4 (l / 16) + e) and m = l % 16, which is how the
// products want the k of a next operand.
__device__ __forceinline__ f64x4 mfma64_k4(double w, double a, f64x4 sums) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(w, a, sums, 0, 0, 0);
}
__device__ __forceinline__ bool not_finite(float v) { return !(fabsf(v) <= 3.4028235e38f); }

template <int DB, bool CH, bool DELTA>
__global__ void __launch_bounds__(256, DELTA && CH && DB == 8 ? 1 : 2)    // (two workgroups a CU: up to 75 KB of LDS and half of the registers each)
chunk_prepare_kernel(const float* __restrict__ qkv, int C, const float* __restrict__ proj, int ld, int b_off, int a_off,
                     const float* __restrict__ A_log, const float* __restrict__ dt_bias,
                     const float* __restrict__ decay, const int2* __restrict__ chunks, float* __restrict__ scratch,
                     int kv_heads, int heads, int V) {
    constexpr int D = 16 * DB, KLD = D + 4, TLD = CHUNK + 4;
    constexpr int NG = CH ? 4 * DB : 1;                       // decays a lane holds of its token
    // (the linear attention's decays multiply single entries of a sum, whose roundings average out)
    using Decay = typename std::conditional<DELTA, double, float>::type;
    // The same LDS twice: first the keys of columns in the order their lanes read them, and B; then G k and -T beta G k, and T beta.
    constexpr int FIRST_USE = CHUNK * (D + TLD), SECOND_USE = DELTA ? CHUNK * (KLD + TLD) : 0;
    __shared__ __attribute__((aligned(16))) float region[FIRST_USE > SECOND_USE ? FIRST_USE : SECOND_USE];
    float* const cols = region;
    float* const b_rows = region + CHUNK * D;
    float* const rows = region;                               // DELTA alone, as are the next three
    float* const solve = region + CHUNK * KLD;                // T beta
    __shared__ __attribute__((aligned(16))) float lower[DELTA ? CHUNK * TLD : 4];        // beta A below the diagonal
    __shared__ __attribute__((aligned(16))) float inverse[DELTA ? 4 * 16 * 20 : 4];      // of I + its diagonal blocks
    __shared__ Decay behind[CH ? 1 : CHUNK];                  // a token's product of decays to its block's end
    __shared__ Decay total[4][CH ? D : 1];                    // a block's product of decays
    __shared__ float betas[CHUNK];
    __shared__ int wild_from, wild_values;
    const int h = blockIdx.x, chunk = blockIdx.y;             // (heads first, as in the other kernel: what it reads lies in its XCD's L2)
    const int first = chunks[chunk].x, n = chunks[chunk].y;
    const ChunkLayout at = chunk_layout(D, V, DELTA);
    float* out = scratch + ((size_t)chunk * heads + h) * at.size;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 15, q = lane >> 4;
    const int kvh = h / (heads / kv_heads);
    const int q_at = kvh * D, k_at = (kv_heads + kvh) * D, v_at = 2 * kv_heads * D + h * V;

    // ---- this wave's 16 tokens: lane (r, q) holds entries 4 s + q of token r
    const int token = 16 * wave + r;
    bool real = token < n;
    const float* row = qkv + (size_t)(first + (real ? token : 0)) * C;
    f32x4 kq[DB], qq[DB];
    Decay pre[NG];
    float beta = 0.f;
    bool wild = false, wild_query = false, wild_value = false;
#pragma unroll
    for (int b = 0; b < DB; ++b) {
        kq[b] = load_quad<true>(row + k_at + 16 * b + 4 * q, 4);
        qq[b] = load_quad<true>(row + q_at + 16 * b + 4 * q, 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) wild |= not_finite(kq[b][e]), wild_query |= not_finite(qq[b][e]);
    }
    for (int v = 4 * q; v < V; v += 16) {
        const f32x4 x = load_quad<true>(row + v_at + v, 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) wild_value |= not_finite(x[e]);
    }
    if (CH) {
        const float* g = decay + ((size_t)(first + (real ? token : 0)) * heads + h) * D + 4 * q;
#pragma unroll
        for (int b = 0; b < DB; ++b) {
            f32x4 x = load_quad<true>(g + 16 * b, 4);
            transpose_quads(x);
#pragma unroll
            for (int e = 0; e < 4; ++e) pre[4 * b + e] = x[e], wild |= not_finite(x[e]);
        }
    } else {
        const float z = proj[(size_t)(first + (real ? token : 0)) * ld + a_off + h] + dt_bias[h];
        const float factor = expf(-expf(A_log[h]) * (z > 20.f ? z : log1pf(expf(z))));
        pre[0] = factor;
        wild |= not_finite(factor);
    }
    if (DELTA) {
        beta = 1.0f / (1.0f + expf(-proj[(size_t)(first + (real ? token : 0)) * ld + b_off + h]));
        wild |= not_finite(beta);
    }
    // What is not finite reaches what it reaches in the walk: a query its own token's output, a value its column from there on, a key,
    // a decay or a beta all of the head from there on (the state too: with a row a key entry that would be lost alone, no
    // later output is without it). It is left out here, and the second kernel makes what comes of it not a number.
    if (tid == 0) wild_from = CHUNK, wild_values = 0;
    __syncthreads();
    if (real && wild) atomicMin(&wild_from, token);
    if (real && wild_value) wild_values = 1;
    unsigned long long lost = __ballot(real && wild_query);
    lost |= lost >> 32;
    lost = (lost | lost >> 16) & 0xffff;
    const bool asks = !((lost >> r) & 1);
    if (lane == 0) ((int*)out)[at.lost + wave] = (int)lost;
    __syncthreads();
    const int from = wild_from;
    const bool screen = wild_values;
    for (int c = tid; c < V; c += 256) {
        int f = from;
        if (screen)
            for (int t = min(n, from) - 1; t >= 0; --t)
                if (not_finite(qkv[(size_t)(first + t) * C + v_at + c])) f = t;
        ((int*)out)[at.from + c] = f;
    }
    real = real && token < from;
    Decay suf[NG];
#pragma unroll
    for (int i = 0; i < NG; ++i) pre[i] = real ? pre[i] : (Decay)1, suf[i] = 1;
    if (!real) beta = 0.f;
    if (q == 0) betas[token] = beta;
    double own = 0.0;                                         // q . k of the token itself
#pragma unroll
    for (int b = 0; b < DB; ++b) {
        if (!real) kq[b] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (!real || !asks) qq[b] = f32x4{0.f, 0.f, 0.f, 0.f};
        transpose_quads(kq[b]);
        transpose_quads(qq[b]);
#pragma unroll
        for (int e = 0; e < 4; ++e) own = fma((double)qq[b][e], (double)kq[b][e], own);
    }
    own += __shfl_xor(own, 16, HB_WAVE);
    own += __shfl_xor(own, 32, HB_WAVE);

    // ---- pairs within the block, level by level; sums lie as (later token 4 e + q, earlier token r). (Sums of the pairs that
    // are not a level's are not used: there is no need to make them zero.)
    f64x4 a_sum = {0.0, 0.0, 0.0, 0.0}, b_sum = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (4 * e + q == r) b_sum[e] = own;
    // With one decay a head the pairs' sums over the key's entries are made once, without decays, and each takes the product of the
    // decays between behind it; with a decay a channel a level's decays are in its operands.
    f64x4 al = {0.0, 0.0, 0.0, 0.0}, bl = al;
    auto pairs = [&]() {
        al = bl = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int i = 0; i < 4 * DB; ++i) {
            const double k = kq[i / 4][i % 4];
            if (DELTA) al = mfma64_k4(k, k, al);
            bl = mfma64_k4(qq[i / 4][i % 4], k, bl);
        }
    };
    if (!CH) pairs();
#pragma unroll
    for (int level = 0; level < 4; ++level) {
        const int s = 1 << level;
        const bool late = (r / s) & 1;
        if (CH) {
            // (the keys and queries are made float64 anew in every level: kept so they would take twice their registers)
#pragma unroll
            for (int b = 0; b < DB; ++b) asm volatile("" : "+v"(kq[b]), "+v"(qq[b]));
            al = bl = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int i = 0; i < 4 * DB; ++i) {
                const Decay f = late ? pre[CH ? i : 0] : suf[CH ? i : 0];
                const double k = kq[i / 4][i % 4] * f;
                if (DELTA) al = mfma64_k4(k, k, al);
                bl = mfma64_k4(qq[i / 4][i % 4] * f, k, bl);
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int t = 4 * e + q;
            const bool pair = t / (2 * s) == r / (2 * s) && ((t / s) & 1) && !((r / s) & 1);
            const double f = CH ? 1.0 : __shfl(pre[0], (lane & 48) + t, HB_WAVE) * suf[0];
            if (pair) a_sum[e] = CH ? al[e] : al[e] * f, b_sum[e] = CH ? bl[e] : bl[e] * f;
        }
        // the products over runs of 2 s: up to a token from its run's start, and behind a token to its run's end
        const int before = (lane & 48) + (r & ~(2 * s - 1)) + s - 1, after = before + s;
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            const Decay p = pre[i];
            const Decay head = __shfl(p, before, HB_WAVE), tail = __shfl(p, after, HB_WAVE);
            if (late) pre[i] = head * p;
            else suf[i] *= tail;
        }
    }
    if (CH) {
        if (r == 15) {
#pragma unroll
            for (int i = 0; i < NG; ++i) total[wave][4 * i + q] = pre[i];
        }
    } else if (lane == 15) {
        total[wave][0] = pre[0];
    }
#pragma unroll
    for (int b = 0; b < DB; ++b) {
        f32x4 k = kq[b];
        if (CH) {
#pragma unroll
            for (int e = 0; e < 4; ++e) k[e] = (float)(kq[b][e] * suf[CH ? 4 * b + e : 0]);
        }
        *(f32x4*)&cols[((wave * DB + b) * 64 + lane) * 4] = k;
    }
    if (!CH && q == 0) behind[CH ? 0 : token] = suf[0];
    auto put = [&](f64x4 a, f64x4 b, int block) {             // sums of (16 wave + 4 e + q, 16 block + r)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int t = 16 * wave + 4 * e + q;
            if (DELTA) lower[t * TLD + in_quads(16 * block + r)] = (float)(betas[t] * a[e]);
            b_rows[t * TLD + in_quads(16 * block + r)] = (float)b[e];
        }
    };
    put(a_sum, b_sum, wave);
    __syncthreads();
    double x[DELTA ? 16 : 1];
    if (DELTA) {
        // the inverse of I + the diagonal block: column r of it, by substitution (the four lane rows do the same)
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            double v = t == r ? 1.0 : 0.0;
#pragma unroll
            for (int i = 0; i < t; ++i) v = fma(-(double)lower[(16 * wave + t) * TLD + in_quads(16 * wave + i)], x[i], v);
            x[t] = v;
        }
#pragma unroll
        for (int t = 0; t < 16; ++t)
            if ((t & 3) == q) inverse[(16 * wave + t) * 20 + in_quads(r)] = (float)x[t];
    }
    // ---- pairs with earlier blocks, from the nearest on: the rows' decays grow by a block's product at a time
    for (int block = wave - 1; block >= 0; --block) {
        f64x4 al = {0.0, 0.0, 0.0, 0.0}, bl = al;
#pragma unroll
        for (int b = 0; b < DB; ++b) {
            const f32x4 k = *(const f32x4*)&cols[((block * DB + b) * 64 + lane) * 4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (CH) {
                    const Decay p = pre[CH ? 4 * b + e : 0];
                    if (DELTA) al = mfma64_k4(kq[b][e] * p, k[e], al);
                    bl = mfma64_k4(qq[b][e] * p, k[e], bl);
                    pre[CH ? 4 * b + e : 0] *= total[block][CH ? 16 * b + 4 * e + q : 0];
                } else {
                    if (DELTA) al = mfma64_k4(kq[b][e], k[e], al);
                    bl = mfma64_k4(qq[b][e], k[e], bl);
                }
            }
        }
        if (!CH) {
            const double f = behind[CH ? 0 : 16 * block + r];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const double g = __shfl(pre[0], (lane & 48) + 4 * e + q, HB_WAVE) * f;
                al[e] *= g, bl[e] *= g;
            }
            pre[0] *= total[block][0];
        }
        put(al, bl, block);
    }
    f32x4 gk[DELTA ? DB : 1];                                 // G k
#pragma unroll
    for (int b = 0; b < DB; ++b) {
        f32x4 gq;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const Decay p = pre[CH ? 4 * b + e : 0];
            gq[e] = (float)(qq[b][e] * p);
            if (DELTA) gk[b][e] = (float)(kq[b][e] * p);
        }
        *(f32x4*)(out + at.q + ((wave * DB + b) * 64 + lane) * 4) = gq;
    }
    // behind a token to the chunk's end
    for (int block = wave + 1; block < 4; ++block) {
#pragma unroll
        for (int i = 0; i < NG; ++i) suf[i] *= CH ? total[block][4 * i + q] : total[block][0];
    }
    // (blocks above the diagonal are never read: a token's row of B goes out up to its own block)
#pragma unroll
    for (int b = 0; b < 4; ++b)
        if (b <= wave)
            *(f32x4*)(out + at.b + ((wave * 4 + b) * 64 + lane) * 4) = *(const f32x4*)&b_rows[(16 * wave + r) * TLD + 16 * b + 4 * q];
    if (CH) {
        for (int d = tid; d < D; d += 256) out[at.g + d] = total[0][d] * total[1][d] * total[2][d] * total[3][d];
    } else {
        for (int d = tid; d < D; d += 256) out[at.g + d] = (float)(total[0][0] * total[1][0] * total[2][0] * total[3][0]);
    }
    __syncthreads();                                          // cols and B have been read
    // G_64 / G k with a row a key entry: a block of 16 tokens and 16 entries at a time, turned in LDS of the wave's own
    float* const turn = (DELTA ? solve : region) + wave * 16 * 20;
#pragma unroll
    for (int b = 0; b < DB; ++b) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            turn[(4 * e + q) * 20 + in_quads(r)] = (float)(kq[b][e] * suf[CH ? 4 * b + e : 0]);
            if (DELTA) rows[token * KLD + in_quads(16 * b + 4 * e + q)] = gk[b][e];
        }
        asm volatile("" ::: "memory");                        // (a wave's LDS accesses keep their order)
        *(f32x4*)(out + at.k + ((b * 4 + wave) * 64 + lane) * 4) = *(const f32x4*)&turn[r * 20 + 4 * q];
        asm volatile("" ::: "memory");
    }
    if (!DELTA) return;
    __syncthreads();                                          // turn has been read

    // ---- T beta, a block of 16 columns a wave: its blocks of rows one after another, as the next product wants them
    {
        f64x4 t[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) t[0][e] = q == 0 ? x[4 * e] : q == 1 ? x[4 * e + 1] : q == 2 ? x[4 * e + 2] : x[4 * e + 3];
#pragma unroll
        for (int n_below = 0; n_below < 4; ++n_below) {       // (the block of rows wave + n_below)
            const int i = wave + n_below;
            if (i >= 4) break;
            if (n_below > 0) {
                f64x4 sum = {0.0, 0.0, 0.0, 0.0}, solved = sum;
#pragma unroll
                for (int j = 0; j < n_below; ++j) {
                    const f32x4 l = *(const f32x4*)&lower[(16 * i + r) * TLD + 16 * (wave + j) + 4 * q];
#pragma unroll
                    for (int s = 0; s < 4; ++s) sum = mfma64_k4(l[s], t[j][s], sum);
                }
                const f32x4 inv = *(const f32x4*)&inverse[(16 * i + r) * 20 + 4 * q];
#pragma unroll
                for (int s = 0; s < 4; ++s) solved = mfma64_k4(inv[s], -sum[s], solved);
                t[n_below] = solved;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
                solve[(16 * i + 4 * e + q) * TLD + in_quads(16 * wave + r)] = (float)(t[n_below][e] * betas[16 * wave + r]);
        }
    }
    __syncthreads();
    // ---- and applied to [G K | V], 16 columns at a time
    for (int cb = wave; cb < DB + V / 16; cb += 4) {
        const bool of_k = cb < DB;
        f32x4 y[4];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = 16 * j + 4 * e + q;
                float v = 0.f;
                if (of_k) v = rows[t * KLD + in_quads(16 * cb + r)];
                else if (t < n && t < from) v = qkv[(size_t)(first + t) * C + v_at + 16 * (cb - DB) + r];
                if (screen && not_finite(v)) v = 0.f;
                y[j][e] = v;
            }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j <= i; ++j) {
                const f32x4 w = *(const f32x4*)&solve[(16 * i + r) * TLD + 16 * j + 4 * q];
#pragma unroll
                for (int s = 0; s < 4; ++s) sum = mfma_k4(w[s], y[j][s], sum);
            }
            if (of_k) {
#pragma unroll
                for (int e = 0; e < 4; ++e) rows[(16 * i + 4 * q + e) * KLD + in_quads(16 * cb + r)] = -sum[e];
            } else {
                *(f32x4*)(out + at.u + ((i * (V / 16) + cb - DB) * 64 + lane) * 4) = sum;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int b = 0; b < DB; ++b)
        *(f32x4*)(out + at.w + ((wave * DB + b) * 64 + lane) * 4) = *(const f32x4*)&rows[(16 * wave + r) * KLD + 16 * b + 4 * q];
}

// Eight waves: four on the chain (a block of 16 tokens of U, then a quarter of the state's rows), four on the outputs (a block of 16 tokens),
// which nothing waits for: they follow a phase behind the chain, in the gaps that it leaves the matrix cores (a chunk of a head of 128 x 128: chain
// 64 products of 32 cycles, 0.9 us, with the two exchanges 1.8, outputs 48). One sequence of 2,048 tokens, 16 heads of 128 x 128: 99 us, by four
// waves that did both, one after the other, 118 (110 with this loop).
template <int DB, bool DELTA>
__global__ void __launch_bounds__(512)
chunk_scan_kernel(const float* __restrict__ qkv, int C, const float* __restrict__ scratch, float* __restrict__ state,
                  const int4* __restrict__ runs, const int* __restrict__ slots, float* __restrict__ out,
                  int kv_heads, int heads, int V, float out_scale) {
    constexpr int D = 16 * DB, OWN = DB / 4;                  // blocks of 16 of the state's rows a wave owns
    constexpr int SLD = D + 4, ULD = CHUNK + 4;
    __shared__ __attribute__((aligned(16))) float s_lds[2][16 * SLD], u_lds[2][16 * ULD];
    const int h = blockIdx.x, vb = blockIdx.y;
    const int4 run = runs[blockIdx.z];
    const int begin = run.z, n_all = run.w, last = (n_all + CHUNK - 1) / CHUNK;
    if (last <= 0) return;
    const ChunkLayout at = chunk_layout(D, V, DELTA);
    const float* part = scratch + ((size_t)run.y * heads + h) * at.size;
    const size_t chunk_step = (size_t)heads * at.size;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6) & 3;
    const bool chain = __builtin_amdgcn_readfirstlane(tid >> 6) < 4;
    const int r = lane & 15, q = lane >> 4;
    const int col = 16 * vb + r;
    // (every load is made, of a place at hand where there is none: with loads that may be left out the compiler waits for all that are in
    // flight at the first use of any)
    auto values = [&](int c, float* v) {
        const int n = n_all - c * CHUNK;
        const float* from = qkv + (size_t)(begin + c * CHUNK) * C + 2 * kv_heads * D + h * V + col;
#pragma unroll
        for (int s = 0; s < 16; ++s) v[s] = from[(size_t)(4 * s + q < n ? 4 * s + q : n - 1) * C];
    };
    // u of a chunk's tokens, as the products want them: without a correction the values themselves
    auto tokens = [&](int c, int buf, const float* v, int from, f32x4* us) {
        if (DELTA) {
#pragma unroll
            for (int b = 0; b < 4; ++b) us[b] = *(const f32x4*)&u_lds[buf][r * ULD + 16 * b + 4 * q];
            return;
        }
#pragma unroll
        for (int b = 0; b < 4; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = 16 * b + 4 * e + q;
                us[b][e] = t < from && c * CHUNK + t < n_all ? v[4 * b + e] : 0.f;
            }
    };

    // Barriers of a chunk: one when u lies in LDS (with a correction), one when the next state does.
    if (chain) {
        struct Operands {
            f32x4 w[DELTA ? DB : 1], k[OWN][4], u, g[OWN];
            float v[DELTA ? 1 : 16];
            int from;
        };
        auto fetch = [&](int c, Operands& o) {
            const float* p = part + (size_t)c * chunk_step;
            if (DELTA) {
#pragma unroll
                for (int b = 0; b < DB; ++b) o.w[b] = *(const f32x4*)(p + at.w + ((wave * DB + b) * 64 + lane) * 4);
                o.u = *(const f32x4*)(p + at.u + ((wave * (V / 16) + vb) * 64 + lane) * 4);
            } else {
                values(c, o.v);
            }
#pragma unroll
            for (int i = 0; i < OWN; ++i) {
                o.g[i] = *(const f32x4*)(p + at.g + 16 * (wave + 4 * i) + 4 * q);
#pragma unroll
                for (int s = 0; s < 4; ++s) o.k[i][s] = *(const f32x4*)(p + at.k + (((wave + 4 * i) * 4 + s) * 64 + lane) * 4);
            }
            o.from = ((const int*)p)[at.from + col];
        };
        float* S_mem = state + ((size_t)slots[run.x] * heads + h) * D * V + col;
        f32x4 S[OWN];
        auto share = [&](int buf) {
#pragma unroll
            for (int i = 0; i < OWN; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) s_lds[buf][r * SLD + 16 * (wave + 4 * i) + 4 * e + q] = S[i][e];
        };
        auto step = [&](int c, int buf, const Operands& o, Operands& next) {
            fetch(c + 1 < last ? c + 1 : c, next);
            __builtin_amdgcn_sched_barrier(0);
            if (DELTA) {
                Chains<8> uc;
#pragma unroll
                for (int b = 0; b < DB; ++b) {
                    const f32x4 s = *(const f32x4*)&s_lds[buf][r * SLD + 16 * b + 4 * q];
#pragma unroll
                    for (int e = 0; e < 4; ++e) uc.add(o.w[b][e], s[e], 4 * b + e);
                }
                const f32x4 u = o.u + uc.sum();
#pragma unroll
                for (int e = 0; e < 4; ++e) u_lds[buf][r * ULD + 16 * wave + 4 * e + q] = u[e];
                hb_workgroup_barrier();
            }
            f32x4 us[4];
            tokens(c, buf, o.v, o.from, us);
            // The state (and the outputs) token by token in ascending order behind what the state before gives, so that the latest tokens,
            // mostly the largest, are added last: as the walk rounds, without its decay of every token.
#pragma unroll
            for (int i = 0; i < OWN; ++i) S[i] *= o.g[i];
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int i = 0; i < OWN; ++i) S[i] = mfma_k4(o.k[i][b][e], us[b][e], S[i]);
            if (o.from < CHUNK) {
#pragma unroll
                for (int i = 0; i < OWN; ++i) S[i] = f32x4{NAN, NAN, NAN, NAN};
            }
            share(buf ^ 1);
            hb_workgroup_barrier();
        };
        __builtin_amdgcn_s_setprio(3);
        Operands even, odd;
        fetch(0, even);                                       // (asked for before the state, whose slot is a load away)
#pragma unroll
        for (int i = 0; i < OWN; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) S[i][e] = S_mem[(size_t)(16 * (wave + 4 * i) + 4 * q + e) * V];
        share(0);
        hb_workgroup_barrier();
        for (int c = 0; c < last; c += 2) {                   // (two by two: the operands' registers take turns, nothing is copied)
            step(c, 0, even, odd);
            if (c + 1 < last) step(c + 1, 1, odd, even);
        }
#pragma unroll
        for (int i = 0; i < OWN; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) S_mem[(size_t)(16 * (wave + 4 * i) + 4 * q + e) * V] = S[i][e];
        return;
    }

    struct Operands {
        f32x4 qg[DB], b[4];
        float v[DELTA ? 1 : 16];
        int from, lost;
    };
    auto fetch = [&](int c, Operands& o) {
        const float* p = part + (size_t)c * chunk_step;
#pragma unroll
        for (int b = 0; b < DB; ++b) o.qg[b] = *(const f32x4*)(p + at.q + ((wave * DB + b) * 64 + lane) * 4);
#pragma unroll
        for (int b = 0; b < 4; ++b) o.b[b] = *(const f32x4*)(p + at.b + ((wave * 4 + (b <= wave ? b : wave)) * 64 + lane) * 4);
        if (!DELTA) values(c, o.v);
        o.from = ((const int*)p)[at.from + col];
        o.lost = ((const int*)p)[at.lost + wave];
    };
    f32x4 held;                                               // a chunk's outputs, on their way before the next but one chunk's loads
    auto leave = [&](int c) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int at_token = c * CHUNK + 16 * wave + 4 * q + e;
            if (c >= 0 && at_token < n_all) out[(size_t)(begin + at_token) * heads * V + h * V + col] = held[e];
        }
    };
    // What the chain holds in LDS for chunk c: the state until u of the chunk after it is there, u until the state after that one is. So with a
    // correction the outputs' products begin once u of their own chunk is there and end in the chunk after it.
    constexpr int FIRST = DELTA ? 3 * DB / 4 : DB;
    auto step = [&](int c, int buf, const Operands& o, Operands& next) {
        if (DELTA) hb_workgroup_barrier();
        leave(c - 1);
        fetch(c + 1 < last ? c + 1 : c, next);
        __builtin_amdgcn_sched_barrier(0);
        Chains<8> oc;
        auto of_state = [&](int b) {
            const f32x4 s = *(const f32x4*)&s_lds[buf][r * SLD + 16 * b + 4 * q];
#pragma unroll
            for (int e = 0; e < 4; ++e) oc.add(o.qg[b][e], s[e], 4 * b + e);
        };
#pragma unroll
        for (int b = 0; b < FIRST; ++b) of_state(b);
        if (DELTA) hb_workgroup_barrier();
#pragma unroll
        for (int b = FIRST; b < DB; ++b) of_state(b);
        f32x4 us[4];
        tokens(c, buf, o.v, o.from, us);
        f32x4 sums = oc.sum();
#pragma unroll
        for (int b = 0; b < 4; ++b)
            if (b <= wave) {
#pragma unroll
                for (int e = 0; e < 4; ++e) sums = mfma_k4(o.b[b][e], us[b][e], sums);
            }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            held[e] = 16 * wave + 4 * q + e < o.from && !(o.lost >> (4 * q + e) & 1) ? sums[e] * out_scale : NAN;
        if (!DELTA) hb_workgroup_barrier();
    };
    Operands even, odd;
    fetch(0, even);
    hb_workgroup_barrier();
    for (int c = 0; c < last; c += 2) {
        step(c, 0, even, odd);
        if (c + 1 < last) step(c + 1, 1, odd, even);
    }
    leave(last - 1);
}

// As hb_gated_delta of recurrent.hip, for keys of 64 or 128 and values in steps of 16, rows in whole quads, and for those
// sequences only that its lists name. chunks [n_chunks]: the row of the chunk's first token, and its tokens (1 to 64).
// runs [n_runs]: the sequence, the place of its first chunk in `chunks` (the others follow), the row of its first token and
// the tokens that its chunks hold (all but the last hold 64). scratch holds n_chunks x heads parts of chunk_floats
// (chunk_layout's size). A sequence longer than the scratch goes through in several calls, its state carried in `state`.
extern "C" int hb_chunked_delta(const float* qkv, int C, const float* proj, int ld, int b_off, int a_off, const float* A_log,
                                const float* dt_bias, const float* decay, float* state, const int* chunks, int n_chunks,
                                const int* runs, int n_runs, const int* slots, float* out, float* scratch, int kv_heads,
                                int heads, int D, int V, int correction, float out_scale, int chunk_floats,
                                hipStream_t stream) {
    HB_REQUIRE(correction || decay, "linear attention: a decay a key channel must be given");
    HB_REQUIRE(n_chunks > 0 && n_runs > 0 && heads > 0 && kv_heads > 0 && heads % kv_heads == 0, "delta rule: %d heads on %d key heads", heads, kv_heads);
    HB_REQUIRE((D == 64 || D == 128) && V > 0 && V % 16 == 0, "delta rule in chunks: keys of %d, values of %d", D, V);
    HB_REQUIRE(C >= 2 * kv_heads * D + heads * V && C % 4 == 0 && (uintptr_t)qkv % 16 == 0 && (uintptr_t)decay % 16 == 0 &&
               (uintptr_t)scratch % 16 == 0, "delta rule in chunks: rows of %d are not in whole quads", C);
    HB_REQUIRE((uintptr_t)chunks % 8 == 0 && (uintptr_t)runs % 16 == 0, "delta rule in chunks: the lists are not aligned");
    HB_REQUIRE(chunk_floats == chunk_layout(D, V, correction != 0).size,
               "delta rule in chunks: a part of %d floats is not the kernel's layout", chunk_floats);
    HB_REQUIRE(n_runs <= 65535 && n_chunks <= 65535 && V / 16 <= 65535, "delta rule: too many sequences or heads for the grid");
    const dim3 grid(heads, n_chunks), scan(heads, V / 16, n_runs);
#define HB_CHUNKS(DB, CH, DELTA)                                                                                      \
    do {                                                                                                              \
        chunk_prepare_kernel<DB, CH, DELTA><<<grid, 256, 0, stream>>>(qkv, C, proj, ld, b_off, a_off, A_log, dt_bias,  \
            decay, (const int2*)chunks, scratch, kv_heads, heads, V);                                                 \
        HB_CHECK_LAUNCH("chunk_prepare");                                                                             \
        chunk_scan_kernel<DB, DELTA><<<scan, 512, 0, stream>>>(qkv, C, scratch, state, (const int4*)runs, slots, out, \
            kv_heads, heads, V, out_scale);                                                                           \
    } while (0)
    if (D == 128 && !correction) HB_CHUNKS(8, true, false);
    else if (D == 128 && decay) HB_CHUNKS(8, true, true);
    else if (D == 128) HB_CHUNKS(8, false, true);
    else if (!correction) HB_CHUNKS(4, true, false);
    else if (decay) HB_CHUNKS(4, true, true);
    else HB_CHUNKS(4, false, true);
#undef HB_CHUNKS
    HB_CHECK_LAUNCH("chunk_scan");
    return 0;
}

// ---------------------------------------------------------------- state-space layer with one decay a head, in chunks
// recurrent.hip has the rule: S <- a S + dt B x^T, y = S^T C + D x, with a = exp(-rate dt), one number a head and token, and B and C
// shared by the heads of a group. With c_t the sum of rate dt up to token t of a chunk,
//   y_t = exp(-c_t) S_0^T C_t + sum_(i<=t) (C_t . B_i) exp(c_i - c_t) dt_i x_i + D x_t
//   S   = exp(-c_64) S_0 + sum_i B_i exp(c_i - c_64) dt_i x_i
// (Dao and Gu, 2024: state-space duality; the sums c and their differences in float64, so that a pair's decay is exact to its
// own size, and no quotient of decays is formed.) Products on the matrix cores, in float32, those of pairs in float64 and rounded once.
// ssm_pairs_kernel: C_t . B_i of a (chunk, group) once for all its heads, as the second kernel's lanes load them.
// A factor beyond TOO_LARGE (inputs, B, C, the state) counts as not finite here: below it no product before its decay passes float32's
// range (sums of 128 products of two are 1.3e38 at most), beyond it one may where the walk, whose state decays first, stays within.
// ssm_chunks_kernel: the chain of chunks, a workgroup a (head, 16 or 32 columns of S, sequence): four waves, each 16 tokens of a chunk for the outputs and a
// quarter of the state's rows. A chunk that holds something not finite is walked token by token instead (ssm_slowly), so that it
// spoils what it spoils in the walk: all its columns, or where an input or the state is what is too large, the 16 columns around it.
// 64 heads of 128 x 64 on 8 groups, one sequence of 2,048 tokens 212 us (the walk 802), of 512 63 (209), four of 512 111 (313), 16 of 128 119
// (310); with a branch on whether a chunk is walked that the compiler took for one a lane 225, 67, 121 and 128. Bound by a chunk's chain in a
// workgroup, 6.3 us with 16 columns, 8.7 with 32: 80 or 160 products of 40 cycles a wave, and as long again
// for the decays and for laying out the state and the columns. Errors against 64 bits are 0.2 to 1.02 of the walk's.
#define TOO_LARGE 1e18f
__device__ __forceinline__ bool too_large(float v) { return !(fabsf(v) <= TOO_LARGE); }

template <int DB>
__global__ void __launch_bounds__(256)
ssm_pairs_kernel(const float* __restrict__ u, int ldu, int b_at, int c_at, const int2* __restrict__ chunks,
                 float* __restrict__ pairs, int groups) {
    constexpr int N = 16 * DB;
    const int g = blockIdx.x, chunk = blockIdx.y;
    const int first = chunks[chunk].x, n = chunks[chunk].y;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, q = lane >> 4;
    auto row_of = [&](int t) { return u + (size_t)(first + min(t, n - 1)) * ldu; };    // (tokens past the end: the last one again, unused)
    f32x4 c[DB];
    const float* c_row = row_of(16 * wave + r) + c_at + g * N + 4 * q;
#pragma unroll
    for (int b = 0; b < DB; ++b) c[b] = load_quad<true>(c_row + 16 * b, 4);
#pragma unroll
    for (int b = 0; b < DB; ++b) transpose_quads(c[b]);
    float* out = pairs + ((size_t)chunk * groups + g) * CHUNK * CHUNK;
    for (int block = 0; block <= wave; ++block) {
        const float* b_row = row_of(16 * block + r) + b_at + g * N + 4 * q;
        f32x4 k[DB];
#pragma unroll
        for (int b = 0; b < DB; ++b) k[b] = load_quad<true>(b_row + 16 * b, 4);
        f64x4 sum = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int b = 0; b < DB; ++b) {
            transpose_quads(k[b]);
#pragma unroll
            for (int e = 0; e < 4; ++e) sum = mfma64_k4(k[b][e], c[b][e], sum);
        }
        // (earlier token 16 block + 4 e + q, later token 16 wave + r)
        const f32x4 s = {(float)sum[0], (float)sum[1], (float)sum[2], (float)sum[3]};
        *(f32x4*)(out + ((wave * 4 + block) * 64 + lane) * 4) = s;
    }
}

// One chunk token by token, of those blocks of 16 of a workgroup's COLS columns whose bit is set; the state lies in LDS, a column's entry n at
// in_quads(n). Eight lanes a column.
template <int N, int SLD, int COLS>
__device__ __forceinline__ void ssm_slowly(int blocks, float* s_lds, const float* u, int ldu, const float* proj, int ld, int n, int x_at, int b_at, int c_at,
                                           float bias, float rate, float skip, float* y, int ldy, int cols) {
    const int col = threadIdx.x / 8, part = threadIdx.x % 8;
    if (col >= COLS || !(blocks >> col / 16 & 1)) return;
    for (int t = 0; t < n; ++t) {
        const float* row = u + (size_t)t * ldu;
        const float z = proj[(size_t)t * ld] + bias, dt = z > 20.f ? z : log1pf(expf(z)), a = expf(-rate * dt);
        const float x = row[x_at + col], dx = dt * x;
        float acc = 0.f;
        for (int i = part * (N / 8); i < (part + 1) * (N / 8); ++i) {
            float& s = s_lds[col * SLD + in_quads(i)];
            s = fmaf(a, s, dx * row[b_at + i]);
            acc = fmaf(s, row[c_at + i], acc);
        }
#pragma unroll
        for (int off = 1; off < 8; off <<= 1) acc += __shfl_xor(acc, off, HB_WAVE);
        if (part == 0 && col < cols) y[(size_t)t * ldy + col] = fmaf(skip, x, acc);
    }
}

template <int DB, int SSM_COLS>
__global__ void __launch_bounds__(256, 2)
ssm_chunks_kernel(const float* __restrict__ u, int ldu, const float* __restrict__ proj, int ld, int dt_off,
                  const float* __restrict__ dt_bias, const float* __restrict__ A_log, const float* __restrict__ Dskip,
                  const float* __restrict__ pairs, float* __restrict__ state, const int4* __restrict__ runs,
                  const int* __restrict__ slots, float* __restrict__ y, int heads, int groups, int P) {
    constexpr int N = 16 * DB, OWN = DB / 4, CB = SSM_COLS / 16;
    constexpr int SLD = N + 4, XLD = CHUNK + 4;
    __shared__ __attribute__((aligned(16))) float s_lds[2][SSM_COLS * SLD], x_lds[2][SSM_COLS * XLD];
    __shared__ double c_lds[4][CHUNK];
    __shared__ float dt_lds[4][CHUNK];
    __shared__ int spoilt[2];                                  // a bit a block of 16 columns that is to be walked
    constexpr int EVERY = (1 << CB) - 1;
    const int h = blockIdx.x, col0 = blockIdx.y * SSM_COLS, cols = min(SSM_COLS, P - col0);
    const int4 run = runs[blockIdx.z];
    const int begin = run.z, n_all = run.w, last = (n_all + CHUNK - 1) / CHUNK;
    const int g = h / (heads / groups), inner = heads * P;
    const int x_at = h * P + col0, b_at = inner + g * N, c_at = inner + (groups + g) * N;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = lane & 15, q = lane >> 4;
    const float rate = expf(A_log[h]), bias = dt_bias[h], skip = Dskip[h];
    // the walk keeps a column's N entries side by side
    float* S_mem = state + ((size_t)slots[run.x] * heads + h) * P * N + (size_t)col0 * N;
    f32x4 S[OWN][CB];
#pragma unroll
    for (int i = 0; i < OWN; ++i)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
            S[i][cb] = 16 * cb < cols ? *(const f32x4*)(S_mem + (size_t)(16 * cb + r) * N + 16 * (wave + 4 * i) + 4 * q) : f32x4{0.f, 0.f, 0.f, 0.f};
    auto share = [&](int buf) {
#pragma unroll
        for (int i = 0; i < OWN; ++i)
#pragma unroll
            for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                for (int e = 0; e < 4; ++e) s_lds[buf][(16 * cb + r) * SLD + 16 * (wave + 4 * i) + 4 * e + q] = S[i][cb][e];
    };
    // a chunk's inputs that all waves share: thread tid brings a quarter of token tid / 4's columns (those past the head's are zeros)
    constexpr int XQ = SSM_COLS / 16;                          // in quads
    const int my_token = tid / 4, my_col = tid % 4 * 4 * XQ;
    f32x4 x_next[XQ];
    float z_next;
    auto fetch = [&](int c) {
        const int n = min(CHUNK, n_all - c * CHUNK);
        const float* row = u + (size_t)(begin + c * CHUNK + my_token) * ldu + x_at + my_col;
#pragma unroll
        for (int i = 0; i < XQ; ++i)
            x_next[i] = my_token < n && my_col + 4 * i < cols ? *(const f32x4*)(row + 4 * i) : f32x4{0.f, 0.f, 0.f, 0.f};
        z_next = lane < n ? proj[(size_t)(begin + c * CHUNK + lane) * ld + dt_off + h] : 0.f;
    };
    // ... into LDS: the columns as a product wants a column's tokens, and every wave its own copy of the step sizes and their sums
    auto place = [&](int c, int buf) {
        const int n = min(CHUNK, n_all - c * CHUNK);
        const float z = z_next + bias;
        const float dt = lane < n ? (z > 20.f ? z : log1pf(expf(z))) : 0.f;
        double sum = lane < n ? (double)(rate * dt) : 0.0;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const double o = __shfl_up(sum, off, HB_WAVE);
            if (lane >= off) sum += o;
        }
        c_lds[wave][lane] = sum;
        dt_lds[wave][lane] = dt;
        const float my_dt = __shfl(dt, my_token & 63, HB_WAVE);
        bool bad = false;
#pragma unroll
        for (int i = 0; i < XQ; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                bad |= too_large(x_next[i][e]) || too_large(x_next[i][e] * my_dt);
                x_lds[buf][(my_col + 4 * i + e) * XLD + in_quads(my_token)] = x_next[i][e];
            }
        const int blocks = (not_finite(dt) || not_finite((float)sum) ? EVERY : 0) | (bad ? 1 << my_col / 16 : 0);
        if (blocks) atomicOr(&spoilt[buf], blocks);
    };
    // what a wave reads of a chunk for itself: its 16 tokens of C and their pairs, all tokens' B for its rows of the state
    f32x4 cq[DB], pr[4];
    float k[OWN][16];
    auto ask = [&](int c) {
        const int n = min(CHUNK, n_all - c * CHUNK), t0 = begin + c * CHUNK;
        const float* c_row = u + (size_t)(t0 + min(16 * wave + r, n - 1)) * ldu + c_at + 4 * q;
#pragma unroll
        for (int b = 0; b < DB; ++b) cq[b] = load_quad<true>(c_row + 16 * b, 4);
        const float* p = pairs + ((size_t)(run.y + c) * groups + g) * CHUNK * CHUNK;
#pragma unroll
        for (int b = 0; b < 4; ++b) pr[b] = b <= wave ? *(const f32x4*)(p + ((wave * 4 + b) * 64 + lane) * 4) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            const float* b_row = u + (size_t)(t0 + min(4 * s + q, n - 1)) * ldu + b_at + r;
#pragma unroll
            for (int i = 0; i < OWN; ++i) k[i][s] = b_row[16 * (wave + 4 * i)];
        }
    };
    if (tid < 2) spoilt[tid] = 0;
    fetch(0);
    ask(0);
    share(0);
    __syncthreads();
    place(0, 0);
    __syncthreads();
    for (int c = 0; c < last; ++c) {
        const int buf = c & 1, n = min(CHUNK, n_all - c * CHUNK), t0 = begin + c * CHUNK;
        const bool more = c + 1 < last;
        if (more) fetch(c + 1);
        bool bad = false, large[CB] = {};
#pragma unroll
        for (int b = 0; b < DB; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) bad |= too_large(cq[b][e]);
#pragma unroll
        for (int s = 0; s < 16; ++s)
#pragma unroll
            for (int i = 0; i < OWN; ++i) bad |= too_large(k[i][s]);
#pragma unroll
        for (int i = 0; i < OWN; ++i)
#pragma unroll
            for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                for (int e = 0; e < 4; ++e) large[cb] |= too_large(S[i][cb][e]);
        int blocks = __any(bad) ? EVERY : 0;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) blocks |= __any(large[cb]) ? 1 << cb : 0;
        if (blocks && lane == 0) atomicOr(&spoilt[buf], blocks);
        // the decays: of a token from the chunk's start, of a pair, and to the chunk's end
        const double own = c_lds[wave][16 * wave + r], end = c_lds[wave][CHUNK - 1];
        float from_start[4], to_end[16], dt[16];
#pragma unroll
        for (int e = 0; e < 4; ++e) from_start[e] = expf((float)-c_lds[wave][16 * wave + 4 * q + e]);
        const float all = expf((float)-end);
#pragma unroll
        for (int s = 0; s < 16; ++s) {
            const int i = 4 * s + q;
            const double at = c_lds[wave][i];
            dt[s] = dt_lds[wave][i];
            to_end[s] = expf((float)(at - end));
            pr[s / 4][s % 4] *= i <= 16 * wave + r ? expf((float)(at - own)) : 0.f;
        }
        __syncthreads();                                      // (everyone has looked for what is not finite)
        const int walked = __builtin_amdgcn_readfirstlane(spoilt[buf]);
#pragma unroll
        for (int b = 0; b < DB; ++b) transpose_quads(cq[b]);
        auto products = [&](int cb) {
            Chains<8> part;
#pragma unroll
            for (int b = 0; b < DB; ++b) {
                const f32x4 s = *(const f32x4*)&s_lds[buf][(16 * cb + r) * SLD + 16 * b + 4 * q];
#pragma unroll
                for (int e = 0; e < 4; ++e) part.add(cq[b][e], s[e], 4 * b + e);
            }
            f32x4 sums = part.sum();
#pragma unroll
            for (int e = 0; e < 4; ++e) sums[e] *= from_start[e];
#pragma unroll
            for (int i = 0; i < OWN; ++i) S[i][cb] *= all;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                f32x4 x = *(const f32x4*)&x_lds[buf][(16 * cb + r) * XLD + 16 * b + 4 * q];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    x[e] *= dt[4 * b + e];
                    const float late = x[e] * to_end[4 * b + e];
#pragma unroll
                    for (int i = 0; i < OWN; ++i) S[i][cb] = mfma_k4(k[i][4 * b + e], late, S[i][cb]);
                    if (b <= wave) sums = mfma_k4(pr[b][e], x[e], sums);
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = 16 * wave + 4 * q + e;
                if (t < n && 16 * cb < cols)
                    y[(size_t)(t0 + t) * inner + x_at + 16 * cb + r] =
                        fmaf(skip, x_lds[buf][(16 * cb + r) * XLD + in_quads(t)], sums[e]);
            }
        };
        if (!walked) {
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) products(cb);
        } else {                                              // (of two blocks perhaps one: a column's bits do not hang on how many share a workgroup)
            ssm_slowly<N, SLD, SSM_COLS>(walked, s_lds[buf], u + (size_t)t0 * ldu, ldu, proj + (size_t)t0 * ld + dt_off + h, ld, n, x_at, b_at, c_at, bias,
                                         rate, skip, y + (size_t)t0 * inner + x_at, inner, cols);
            __syncthreads();
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
                if (!(walked >> cb & 1)) {
                    products(cb);
                    continue;
                }
#pragma unroll
                for (int i = 0; i < OWN; ++i)
#pragma unroll
                    for (int e = 0; e < 4; ++e) S[i][cb][e] = s_lds[buf][(16 * cb + r) * SLD + 16 * (wave + 4 * i) + 4 * e + q];
            }
        }
        if (more) {
            ask(c + 1);                                       // (on their way while the state and the columns are laid out)
            share(buf ^ 1);
            place(c + 1, buf ^ 1);
        }
        __syncthreads();
        if (tid == 0) spoilt[buf] = 0;                        // (read again two chunks on, behind a barrier)
    }
#pragma unroll
    for (int i = 0; i < OWN; ++i)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
            if (16 * cb < cols) *(f32x4*)(S_mem + (size_t)(16 * cb + r) * N + 16 * (wave + 4 * i) + 4 * q) = S[i][cb];
}

// As hb_ssm_scan of recurrent.hip, for states of 64 or 128 rows and columns in steps of 16, and for those sequences only that its
// lists name (see hb_chunked_delta). pairs holds n_chunks x groups x 64 x 64 floats.
extern "C" int hb_chunked_ssm(const float* u, int ldu, const float* proj, int ld, int dt_off, const float* dt_bias,
                              const float* A_log, const float* Dskip, float* state, const int* chunks, int n_chunks,
                              const int* runs, int n_runs, const int* slots, float* y, float* pairs, int heads, int groups, int N,
                              int P, int state_floats, hipStream_t stream) {
    HB_REQUIRE(n_chunks > 0 && n_runs > 0 && heads > 0 && groups > 0 && heads % groups == 0, "state-space chunks: %d heads in %d groups", heads, groups);
    HB_REQUIRE((N == 64 || N == 128) && P > 0 && P % 16 == 0 && state_floats == N * P, "state-space chunks: a state of %d x %d in %d floats", N, P, state_floats);
    HB_REQUIRE(ldu >= heads * P + 2 * groups * N && ldu % 4 == 0 && (uintptr_t)u % 16 == 0 && (uintptr_t)state % 16 == 0 && (uintptr_t)pairs % 16 == 0,
               "state-space chunks: rows of %d are not in whole quads", ldu);
    HB_REQUIRE(dt_off >= 0 && dt_off + heads <= ld, "state-space chunks: the columns lie outside their rows");
    HB_REQUIRE((uintptr_t)chunks % 8 == 0 && (uintptr_t)runs % 16 == 0, "state-space chunks: the lists are not aligned");
    // 16 columns of the state a workgroup where that many still fit the chip at once, two a CU: half the products in a chunk's chain, the
    // decays once more. 64 heads of 128 x 64 in 8 groups, us by 32 | 16 columns: one sequence of 2,048 tokens (128 workgroups of 32 columns)
    // 290 | 211, of 512 83 | 63, two of 512 and 300 (256) 84 | 70, three of 512 (384) 109 | 125, four (512) 112 | 148, eight of 128 67 | 85.
    const bool narrow = (long long)heads * ((P + 31) / 32) * n_runs <= 256;
    const int tiles = (P + (narrow ? 15 : 31)) / (narrow ? 16 : 32);
    HB_REQUIRE(n_runs <= 65535 && n_chunks <= 65535 && tiles <= 65535, "state-space chunks: too many sequences or columns for the grid");
#define HB_SSM_CHUNKS(DB, COLS)                                                                                              \
    do {                                                                                                                     \
        ssm_pairs_kernel<DB><<<dim3(groups, n_chunks), 256, 0, stream>>>(u, ldu, heads * P, heads * P + groups * N,          \
                                                                         (const int2*)chunks, pairs, groups);                \
        HB_CHECK_LAUNCH("ssm_pairs");                                                                                        \
        ssm_chunks_kernel<DB, COLS><<<dim3(heads, tiles, n_runs), 256, 0, stream>>>(u, ldu, proj, ld, dt_off, dt_bias, A_log, Dskip, \
            pairs, state, (const int4*)runs, slots, y, heads, groups, P);                                                    \
    } while (0)
    if (N == 128 && narrow) HB_SSM_CHUNKS(8, 16);
    else if (N == 128) HB_SSM_CHUNKS(8, 32);
    else if (narrow) HB_SSM_CHUNKS(4, 16);
    else HB_SSM_CHUNKS(4, 32);
#undef HB_SSM_CHUNKS
    HB_CHECK_LAUNCH("ssm_chunks");
    return 0;
}
