// Attention whose keys and values of all heads come from one latent vector a token.
// What a token leaves in the cache is one row [c (rank) | r (rot)]: the normed latent and one
// rotated key part that the heads share. Head h's key is [W_uk,h c | r] and its value W_uv,h c; with
// the query's unrotated part taken through W_uk,h^T beforehand (q' = W_uk,h^T q_h, `rank` numbers) the
// score is (q' . c + q_rot . r) * scale, and sum_j p_j c_j (rank numbers) goes through W_uv,h
// afterwards: the kernels here see one shared "key head" of rank + rot numbers whose first `rank`
// are also its value. Scores, softmax and the weighted sums are float32 whatever the storage.
//
// Pages: row of position p of a slot at page_table[slot * max_pages + p / page_size], pages
// [page, page_size, rank + rot].
#include "common.h"
#include <math.h>

HB_MODULE_ERROR_SLOT()

#define HB_MAX_KEY 1152                     // rank + rot
#define HB_MAX_RANK 1024
#define ACC_REGS (HB_MAX_RANK / HB_WAVE)

// the pair (a, b) at angle t: (a cos - b sin, b cos + a sin)
__device__ __forceinline__ void rotate_pair(float a, float b, float angle, float& ra, float& rb) {
    float s, c;
    sincosf(angle, &s, &c);
    ra = a * c - b * s;
    rb = b * c + a * s;
}

// ---------------------------------------- what a token writes: its cache row and its rotated queries
// down (rows down_ld floats apart, as q's are q_ld apart: both may be columns of one projection's rows)
// [T, rank + rot] float32: the first `rank` RMS-normed with norm_w -> the row's c; the last `rot`
// rotated (the first rot_dims of them: entry i with i + rot_dims / 2, angle pos * inv_freq[i]; the rest
// unchanged) -> the row's r. q [T, H, qd + rot] float32: every head's last `rot` rotated the same way
// into q_full[t, h, rank ...] (q_full [T, H, rank + rot] float32; its first `rank` are written by the
// product with W_uk^T). One block a token.
// Queries that come from a latent of their own are not there yet when the cache's row is written: the kernel then
// runs twice, first with H = 0 and down's neighbour columns q_down [T, q_rank] (rows down_ld apart), which are
// RMS-normed with q_norm_w into c_q [T, q_rank] (the product that makes the queries reads it), then for the queries alone.
template <class TC>
__global__ void latent_write_kernel(const float* __restrict__ down, int down_ld, const float* __restrict__ norm_w,
                                    const float* __restrict__ q, int q_ld, float* __restrict__ q_full,
                                    bf16* __restrict__ q_plain, const float* __restrict__ inv_freq, const int* __restrict__ positions,
                                    const int* __restrict__ seq_of, const int* __restrict__ slots,
                                    const int* __restrict__ page_table, int max_pages, int page_size,
                                    TC* __restrict__ pages, int H, int qd, int rank, int rot, int rot_dims,
                                    float eps, int write_cache, const float* __restrict__ q_down, int q_rank,
                                    const float* __restrict__ q_norm_w, TC* __restrict__ c_q) {
    __shared__ float red[16];
    const int t = blockIdx.x;
    const int pos = positions[t];
    const int half = rot_dims / 2;
    const float p = (float)pos;
    if (write_cache) {
        const float* in = down + (size_t)t * down_ld;
        float ss = 0.f;
        for (int i = threadIdx.x; i < rank; i += blockDim.x) ss = fmaf(in[i], in[i], ss);
        ss = hb_block_sum(ss, red);
        const float inv = 1.0f / sqrtf(ss / (float)rank + eps);
        const int slot = slots[seq_of[t]];
        const int page = page_table[(size_t)slot * max_pages + pos / page_size];
        TC* row = pages + ((size_t)page * page_size + pos % page_size) * (rank + rot);
        for (int i = threadIdx.x; i < rank; i += blockDim.x) row[i] = hb_from_float<TC>(in[i] * inv * norm_w[i]);
        for (int i = threadIdx.x; i < rot; i += blockDim.x) {
            float v = in[rank + i];
            if (i < rot_dims) {
                const int j = i < half ? i : i - half;
                float ra, rb;
                rotate_pair(in[rank + j], in[rank + j + half], p * inv_freq[j], ra, rb);
                v = i < half ? ra : rb;
            }
            row[rank + i] = hb_from_float<TC>(v);
        }
    }
    if (q_down) {
        const float* in = q_down + (size_t)t * down_ld;
        float ss = 0.f;
        for (int i = threadIdx.x; i < q_rank; i += blockDim.x) ss = fmaf(in[i], in[i], ss);
        ss = hb_block_sum(ss, red);
        const float inv = 1.0f / sqrtf(ss / (float)q_rank + eps);
        for (int i = threadIdx.x; i < q_rank; i += blockDim.x)
            c_q[(size_t)t * q_rank + i] = hb_from_float<TC>(in[i] * inv * q_norm_w[i]);
    }
    for (int e = threadIdx.x; e < H * rot; e += blockDim.x) {
        const int h = e / rot, i = e % rot;
        const float* in = q + (size_t)t * q_ld + (size_t)h * (qd + rot) + qd;
        float v = in[i];
        if (i < rot_dims) {
            const int j = i < half ? i : i - half;
            float ra, rb;
            rotate_pair(in[j], in[j + half], p * inv_freq[j], ra, rb);
            v = i < half ? ra : rb;
        }
        q_full[((size_t)t * H + h) * (rank + rot) + rank + i] = v;
    }
    // the unrotated parts once more as bfloat16 [T, H, qd], for a matrix-core product with W_uk^T
    if (q_plain)
        for (int e = threadIdx.x; e < H * qd; e += blockDim.x) {
            const int h = e / qd, i = e % qd;
            q_plain[(size_t)t * H * qd + e] = hb_from_float<bf16>(q[(size_t)t * q_ld + (size_t)h * (qd + rot) + i]);
        }
}

extern "C" int hb_latent_write(const float* down, int down_ld, const float* norm_w, const float* q, int q_ld, float* q_full,
                               void* q_plain, const float* inv_freq, const int* positions, const int* seq_of, const int* slots,
                               const int* page_table, int max_pages, int page_size, void* pages, int dtype, int T,
                               int H, int qd, int rank, int rot, int rot_dims, float eps, int write_cache,
                               const float* q_down, int q_rank, const float* q_norm_w, void* c_q, hipStream_t stream) {
    HB_REQUIRE(!q_down || (q_rank > 0 && q_norm_w && c_q), "latent write: a query latent needs its norm and a place");
    HB_REQUIRE(T > 0 && (H > 0 || (H == 0 && (q_down || write_cache))) && rank > 0 && rot >= 0 && qd >= 0, "latent write: empty input");
    HB_REQUIRE(rot_dims >= 0 && rot_dims <= rot && rot_dims % 2 == 0, "latent write: %d rotated of %d", rot_dims, rot);
    if (dtype == HB_F32)
        latent_write_kernel<float><<<T, 256, 0, stream>>>(down, down_ld, norm_w, q, q_ld, q_full, (bf16*)q_plain, inv_freq, positions, seq_of, slots,
                                                          page_table, max_pages, page_size, (float*)pages, H, qd,
                                                          rank, rot, rot_dims, eps, write_cache, q_down, q_rank, q_norm_w,
                                                          (float*)c_q);
    else if (dtype == HB_BF16)
        latent_write_kernel<bf16><<<T, 256, 0, stream>>>(down, down_ld, norm_w, q, q_ld, q_full, (bf16*)q_plain, inv_freq, positions, seq_of, slots,
                                                         page_table, max_pages, page_size, (bf16*)pages, H, qd,
                                                         rank, rot, rot_dims, eps, write_cache, q_down, q_rank, q_norm_w,
                                                          (bf16*)c_q);
    else
        HB_REQUIRE(false, "latent write: unknown dtype %d", dtype);
    HB_CHECK_LAUNCH("latent_write");
    return 0;
}

// ------------------------------------------------ attention over the latent rows, plain
// One wave a (token, head). The keys a query at position p sees are [0, p]; they are walked in
// chunks of 64 that start at multiples of 64 of the absolute position, with an online softmax, so
// the rounding depends on the positions only, not on how the tokens were cut into steps or batches.
// out[t, h, :rank] = sum_j p_j c_j, times sigmoid(gate[t * gate_ld + h]) if a gate is given (the
// head's output is linear in it, so the gate may be applied before W_uv). With sinks [H] the softmax's
// denominator of head h also holds exp(sinks[h]), unscaled, once, without key or value.
template <class TC, class TO>
__global__ void __launch_bounds__(HB_WAVE)
latent_attention_plain_kernel(const float* __restrict__ q_full, const TC* __restrict__ pages,
                              TO* __restrict__ out, const float* __restrict__ gate, int gate_ld,
                              const int* __restrict__ positions, const int* __restrict__ seq_of,
                              const int* __restrict__ slots, const int* __restrict__ page_table, int max_pages,
                              int page_size, int H, int rank, int rot, float scale, const float* __restrict__ sinks) {
    __shared__ float qs[HB_MAX_KEY];
    __shared__ float ps[HB_WAVE];
    const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
    const int kd = rank + rot;
    const int pos = positions[t];
    const int* pt = page_table + (size_t)slots[seq_of[t]] * max_pages;
    const float* qrow = q_full + ((size_t)t * H + h) * kd;
    for (int d = lane; d < kd; d += HB_WAVE) qs[d] = qrow[d];
    __syncthreads();

    const int hi = pos + 1;
    float m = -INFINITY, l = 0.f;
    if (sinks) m = sinks[h], l = 1.0f;
    float acc[ACC_REGS];
#pragma unroll
    for (int i = 0; i < ACC_REGS; ++i) acc[i] = 0.f;

    for (int c = 0; c < hi; c += HB_WAVE) {
        const int j = c + lane;
        const bool valid = j < hi;
        float s = -INFINITY;
        if (valid) {
            const TC* kr = pages + ((size_t)pt[j / page_size] * page_size + j % page_size) * kd;
            float dot = 0.f;
            for (int d = 0; d < kd; ++d) dot = fmaf(qs[d], hb_to_float(kr[d]), dot);
            s = dot * scale;
        }
        const float m_new = fmaxf(m, hb_wave_max(s));
        const float corr = expf(m - m_new);
        const float p = valid ? expf(s - m_new) : 0.f;
        l = l * corr + hb_wave_sum(p);
        m = m_new;
        __syncthreads();
        ps[lane] = p;
        __syncthreads();
        const int n = hi - c < HB_WAVE ? hi - c : HB_WAVE;
#pragma unroll
        for (int i = 0; i < ACC_REGS; ++i) acc[i] *= corr;
        for (int jj = 0; jj < n; ++jj) {
            const int jv = c + jj;
            const TC* vr = pages + ((size_t)pt[jv / page_size] * page_size + jv % page_size) * kd;
            const float pj = ps[jj];
#pragma unroll
            for (int i = 0; i < ACC_REGS; ++i) {
                const int d = lane + HB_WAVE * i;
                if (d < rank) acc[i] = fmaf(pj, hb_to_float(vr[d]), acc[i]);
            }
        }
    }
    float w = l > 0.f ? 1.0f / l : 0.f;
    if (gate) w *= 1.0f / (1.0f + expf(-gate[(size_t)t * gate_ld + h]));
    TO* orow = out + ((size_t)t * H + h) * rank;
#pragma unroll
    for (int i = 0; i < ACC_REGS; ++i) {
        const int d = lane + HB_WAVE * i;
        if (d < rank) orow[d] = hb_from_float<TO>(acc[i] * w);
    }
}

extern "C" int hb_latent_attention_plain(const float* q_full, const void* pages, void* out, int dtype,
                                         const float* gate, int gate_ld, const int* positions, const int* seq_of,
                                         const int* slots, const int* page_table, int max_pages, int page_size,
                                         int T, int H, int rank, int rot, float scale, const float* sinks,
                                         hipStream_t stream) {
    HB_REQUIRE(T > 0 && H > 0 && H <= 65535, "latent attention: empty input or too many heads");
    HB_REQUIRE(rank > 0 && rank <= HB_MAX_RANK && rot >= 0 && rank + rot <= HB_MAX_KEY,
               "latent attention: a latent of %d + %d, the kernel takes up to %d + %d", rank, rot, HB_MAX_RANK,
               HB_MAX_KEY - HB_MAX_RANK);
    dim3 grid(T, H);
    if (dtype == HB_F32)
        latent_attention_plain_kernel<float, float><<<grid, HB_WAVE, 0, stream>>>(
            q_full, (const float*)pages, (float*)out, gate, gate_ld, positions, seq_of, slots, page_table, max_pages,
            page_size, H, rank, rot, scale, sinks);
    else if (dtype == HB_BF16)
        latent_attention_plain_kernel<bf16, bf16><<<grid, HB_WAVE, 0, stream>>>(
            q_full, (const bf16*)pages, (bf16*)out, gate, gate_ld, positions, seq_of, slots, page_table, max_pages,
            page_size, H, rank, rot, scale, sinks);
    else
        HB_REQUIRE(false, "latent attention: unknown dtype %d", dtype);
    HB_CHECK_LAUNCH("latent_attention_plain");
    return 0;
}

// ------------------------------------------------ the same attention on the matrix cores (bfloat16 rows)
// A wave takes 16 heads of one token (the rows of its matrix products) and a range of the keys, in
// chunks of 32. Scores: S^T = K Q^T, the chunk's rows straight from memory as operands (a lane: one
// key's 8 consecutive numbers), the query (times the scale) in registers as two bfloat16 halves, high
// and low, so that it keeps 16 bits of mantissa (with the high half alone a test with large queries
// lost a digit). The sums are float32, and so are the softmax and its state, which are a lane's own
// (a lane holds scores of one head only). Weighted sums: O^T = V^T P^T
// with the weights again as high and low halves (they are never rounded to 8 bits), and V^T, the
// chunk's first `rank` numbers a key with the keys along a row, written to LDS from the registers
// that hold them as the scores' operands. The 32 keys
// of a product stand in the order in which the scores' lanes hold them (4 g + i of the first block of
// 16, then of the second), so the weights go from the scores' registers into the next product as they
// are. With more than one range a token the unnormalised sums, maxima and denominators go to scratch
// and a second kernel joins them in the ranges' order.
// Sizes: rank and rot multiples of 32; RB >= rank / 16, KSM >= (rank + rot) / 32.
typedef __bf16 la_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 la_bf16x4 __attribute__((ext_vector_type(4)));
typedef float la_f32x4 __attribute__((ext_vector_type(4)));
#define LA_CHUNK 32
#define LA_VT_STRIDE 36          // bfloat16 a row of V^T in LDS: 32 keys and 8 bytes, so rows start at other banks

__device__ __forceinline__ void la_split(float v, __bf16& hi, __bf16& lo) {
    hi = (__bf16)v;
    lo = (__bf16)(v - (float)hi);
}

template <int RB, int KSM>
__global__ void __launch_bounds__(HB_WAVE)
latent_attention_mfma_kernel(const float* __restrict__ q_full, const bf16* __restrict__ pages,
                             bf16* __restrict__ out, float* __restrict__ part_acc, float* __restrict__ part_ml,
                             const float* __restrict__ gate, int gate_ld, const int* __restrict__ positions,
                             const int* __restrict__ seq_of, const int* __restrict__ slots,
                             const int* __restrict__ page_table, int max_pages, int page_size, int H, int rank,
                             int rot, float scale, int splits, int chunks_per_split, const float* __restrict__ sinks) {
    __shared__ __attribute__((aligned(16))) __bf16 Vt[RB * 16 * LA_VT_STRIDE];
    const int HB = (H + 15) / 16;
    const int t = blockIdx.x / HB, hb = blockIdx.x % HB, split = blockIdx.y;
    const int lane = threadIdx.x, n = lane & 15, g = lane >> 4;
    const int h = hb * 16 + n;
    const bool head = h < H;
    const int pos = positions[t];
    const int* pt = page_table + (size_t)slots[seq_of[t]] * max_pages;
    const int kd = rank + rot, KS = kd / 32, rblocks = rank / 16, vsteps = rank / 32;
    __bf16* vt_w = Vt + (8 * g) * LA_VT_STRIDE + n;          // where this lane's numbers of a key go

    la_bf16x8 qh[KSM], ql[KSM];
    {
        const float* qrow = q_full + ((size_t)t * H + (head ? h : H - 1)) * kd + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KSM; ++ks)
            if (ks < KS) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    __bf16 hi, lo;
                    la_split(qrow[32 * ks + e] * scale, hi, lo);
                    qh[ks][e] = hi;
                    ql[ks][e] = lo;
                }
            }
    }
    const int n_chunks = (pos + LA_CHUNK) / LA_CHUNK;            // chunks that hold a key <= pos
    const int c_begin = split * chunks_per_split;
    const int c_end = n_chunks < c_begin + chunks_per_split ? n_chunks : c_begin + chunks_per_split;
    float m = -INFINITY, l = 0.f;
    la_f32x4 acc[RB];
#pragma unroll
    for (int db = 0; db < RB; ++db) acc[db] = la_f32x4{0.f, 0.f, 0.f, 0.f};

    for (int c = c_begin; c < c_end; ++c) {
        const int j0 = c * LA_CHUNK;
        // the chunk's 32 keys lie in one page (pages hold a multiple of 32 positions)
        const bf16* chunk = pages + ((size_t)pt[j0 / page_size] * page_size + j0 % page_size) * kd;
        la_f32x4 s[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            s[kb] = la_f32x4{0.f, 0.f, 0.f, 0.f};
            const bf16* krow = chunk + (size_t)(kb * 16 + n) * kd + 8 * g;
#pragma unroll
            for (int ks = 0; ks < KSM; ++ks)
                if (ks < KS) {
                    const la_bf16x8 kv = *(const la_bf16x8*)(krow + 32 * ks);
                    s[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kv, qh[ks], s[kb], 0, 0, 0);
                    s[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kv, ql[ks], s[kb], 0, 0, 0);
                    // the same numbers are the key's part of V^T: key 16 kb + n, numbers 32 ks + 8 g + e
                    if (ks < vsteps) {
#pragma unroll
                        for (int e = 0; e < 8; ++e) vt_w[(32 * ks + e) * LA_VT_STRIDE + 16 * kb] = kv[e];
                    }
                }
            // (the second block's loads stay behind the first block's products: all of a chunk's rows in
            //  flight at once would not fit the registers beside the sums)
            __builtin_amdgcn_sched_barrier(0);
        }
        // s[kb][i]: key j0 + 16 kb + 4 g + i against head n
        float cmax = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (j0 + 16 * kb + 4 * g + i > pos) s[kb][i] = -INFINITY;
                cmax = fmaxf(cmax, s[kb][i]);
            }
        cmax = fmaxf(cmax, __shfl_xor(cmax, 16, HB_WAVE));
        cmax = fmaxf(cmax, __shfl_xor(cmax, 32, HB_WAVE));
        const float m_new = fmaxf(m, cmax);                     // finite: the chunk holds a key <= pos
        const float corr = expf(m - m_new);
        la_bf16x8 ph, pl;
        float psum = 0.f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float p = expf(s[kb][i] - m_new);
                psum += p;
                __bf16 hi, lo;
                la_split(p, hi, lo);
                ph[4 * kb + i] = hi;
                pl[4 * kb + i] = lo;
            }
        l = l * corr + psum;
        m = m_new;
        // (rescaled every time: a branch around this, for chunks that leave the maximum as it is, made the
        //  compiler spill the sums)
#pragma unroll
        for (int db = 0; db < RB; ++db)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[db][i] *= corr;
        __syncthreads();
#pragma unroll
        for (int db = 0; db < RB; ++db)
            if (db < rblocks) {
                const __bf16* vr = Vt + (db * 16 + n) * LA_VT_STRIDE + 4 * g;
                const uint2 v0 = *(const uint2*)vr, v1 = *(const uint2*)(vr + 16);
                const la_bf16x8 vv = __builtin_bit_cast(la_bf16x8, uint4{v0.x, v0.y, v1.x, v1.y});
                acc[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vv, ph, acc[db], 0, 0, 0);
                acc[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vv, pl, acc[db], 0, 0, 0);
                if (db % 8 == 7) __builtin_amdgcn_sched_barrier(0);      // (no more than eight blocks' reads in flight)
            }
        __syncthreads();
    }
    l += __shfl_xor(l, 16, HB_WAVE);
    l += __shfl_xor(l, 32, HB_WAVE);
    if (!head) return;
    // acc[db][i]: number 16 db + 4 g + i of head n's sum
    const size_t row = (size_t)t * H + h;
    if (splits == 1) {
        if (sinks) l += expf(sinks[h] - m);                 // (an infinite share, a sink far above every score, leaves 0)
        float w = l > 0.f ? 1.0f / l : 0.f;
        if (gate) w *= 1.0f / (1.0f + expf(-gate[(size_t)t * gate_ld + h]));
#pragma unroll
        for (int db = 0; db < RB; ++db)
            if (db < rblocks) {
#pragma unroll
                for (int i = 0; i < 4; ++i) out[row * rank + db * 16 + 4 * g + i] = hb_from_float<bf16>(acc[db][i] * w);
            }
    } else {
        float* pa = part_acc + (row * splits + split) * rank;
#pragma unroll
        for (int db = 0; db < RB; ++db)
            if (db < rblocks) *(la_f32x4*)(pa + db * 16 + 4 * g) = acc[db];
        if (g == 0) {
            part_ml[(row * splits + split) * 2] = m;
            part_ml[(row * splits + split) * 2 + 1] = l;
        }
    }
}

// ------------------------------------------------ the same for prompts: 64 rows share their keys
// A workgroup takes 64 (token, head) rows of a sequence, head by head and token by token as they lie, and walks the keys that
// any of them sees in chunks of 32. A chunk comes into LDS once for all of them (16 bytes a thread and load, asked for while the
// chunk before is worked on), as operands of the scores and, transposed on the way (four keys of eight numbers a thread,
// eight bytes a write), as operands of the weighted sums. Two waves on every 16 rows: each takes half of a row's numbers
// in the scores (the halves meet in LDS, added in one order by both) and half of the rank in the sums, so that the
// query's two bfloat16 halves (72 registers) and the sums (64) of a wave fit beside a second wave on its SIMD. Operands,
// halves and order of keys are latent_attention_mfma_kernel's; the softmax runs in powers of two, and its reference moves
// only where a weight would pass 2^LP_SLACK. A chunk that a row does not see leaves it as it was, also where its numbers are
// not finite; keys behind the last that a row sees are zeros.
// 2,048 tokens of 16 heads, 512 + 64, take 286 us (a wave a token's 16 heads, keys from the L2s and V transposed by every
// wave: 974), three prompts of 840 to 1,400 tokens 324 (829). Bound by the phases of a chunk (8,500 cycles), which the
// barriers keep apart: LDS is busy for 3,700 of them (1,800 are writes that meet in a bank), the matrix cores for 2,200,
// the vector units for 1,900.
#define LP_ROWS 64
#define LP_SLACK 8.0f
#define LP_LOG2E 1.4426950408889634f
template <int RBW, int KSW>
__global__ void __launch_bounds__(512)
latent_attention_prompt_kernel(const float* __restrict__ q_full, const bf16* __restrict__ pages, bf16* __restrict__ out,
                               const float* __restrict__ gate, int gate_ld, const int* __restrict__ positions,
                               const int* __restrict__ seq_starts, const int* __restrict__ slots,
                               const int* __restrict__ page_table, int max_pages, int page_size, int H, int rank,
                               int rot, float scale, const float* __restrict__ sinks) {
    // operands of 64 lanes x 16 bytes, lane (n, g) at 16 g + (n + a rotation by the operand's number) % 16: reads meet no
    // bank twice, and the writes of threads that hold a key's neighbouring numbers spread over the banks
    __shared__ __attribute__((aligned(16))) uint4 keys[2][2][KSW][HB_WAVE];         // [block of 16 keys][half][32 numbers]
    __shared__ __attribute__((aligned(16))) uint4 Vt[2][2][RBW][HB_WAVE];           // [buffer][half][16 numbers], 32 keys
    __shared__ __attribute__((aligned(16))) la_f32x4 halves[8][2][HB_WAVE];
    __shared__ __attribute__((aligned(16))) int lost_from[32 * RBW];                // [number]: the key from which on it is not finite
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int n = lane & 15, g = lane >> 4, half = wave & 1;
    const int kd = rank + rot, KS = kd / 32, vsteps = rank / 8;
    const int ks_a = (KS + 1) / 2, db_a = (rank / 16 + 1) / 2;              // the first half's steps and blocks
    const int seq = blockIdx.y, tile = gridDim.x - 1 - blockIdx.x;          // (the tiles with the most keys first)
    const int begin = seq_starts[seq], rows = (seq_starts[seq + 1] - begin) * H;
    if (tile * LP_ROWS >= rows) return;
    const int in_seq = tile * LP_ROWS + 16 * (wave >> 1) + n;
    const bool mine = in_seq < rows;
    const int t = begin + (mine ? in_seq : rows - 1) / H, h = (mine ? in_seq : rows - 1) % H;
    const int sees = mine ? positions[t] : -1;                              // the last key that this lane's row sees
    const int pos_first = positions[begin + tile * LP_ROWS / H];
    const int pos_last = positions[begin + min(tile * LP_ROWS + LP_ROWS - 1, rows - 1) / H];
    const int* pt = page_table + (size_t)slots[seq] * max_pages;
    const int n_chunks = pos_last / LA_CHUNK + 1;
    // this wave's share of the scores' steps and of the sums' blocks. (Steps beyond it are zeros in LDS against a query
    // of zeros, blocks beyond it go into sums that go nowhere: there is no branch between the products.)
    const int ks0 = half ? ks_a : 0, ks_n = half ? KS - ks_a : ks_a;
    const int db0 = half ? db_a : 0, db_n = half ? rank / 16 - db_a : db_a;
    for (int i = tid; i < 4 * KSW * HB_WAVE; i += 512) (&keys[0][0][0][0])[i] = uint4{0, 0, 0, 0};
    for (int i = tid; i < 32 * RBW; i += 512) lost_from[i] = 0x7fffffff;

    la_bf16x8 qh[KSW], ql[KSW];
    {
        const float* qrow = q_full + ((size_t)t * H + h) * kd + 32 * ks0 + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KSW; ++ks) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                __bf16 hi, lo;
                la_split(ks < ks_n ? qrow[32 * ks + e] * (scale * LP_LOG2E) : 0.f, hi, lo);
                qh[ks][e] = hi;
                ql[ks][e] = lo;
            }
        }
    }
    float m = -INFINITY, l = 0.f;
    la_f32x4 acc[RBW];
#pragma unroll
    for (int db = 0; db < RBW; ++db) acc[db] = la_f32x4{0.f, 0.f, 0.f, 0.f};

    // a thread's share of a chunk: four keys of eight numbers of the latent, and eight of the rotated part of one
    const int x = tid % vsteps, kg = tid / vsteps;
    const int rx = rot ? tid % (rot / 8) : 0, rkey = rot ? tid / (rot / 8) : LA_CHUNK;
    const int lat_at = 4 * kg * kd + 8 * x, turned_at = rkey * kd + rank + 8 * rx;
    uint4 lat[4], turned;
    auto fetch = [&](int c, int page) {
        const int j0 = c * LA_CHUNK;
        const bf16* chunk = pages + ((size_t)page * page_size + j0 % page_size) * kd;
        if (kg < 8) {
#pragma unroll
            for (int i = 0; i < 4; ++i) lat[i] = *(const uint4*)(chunk + lat_at + i * kd);
        }
        if (rkey < LA_CHUNK) turned = *(const uint4*)(chunk + turned_at);
        if (j0 + LA_CHUNK - 1 > pos_last) {                          // (a page's rows exist whether a token lies there or not)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (j0 + 4 * kg + i > pos_last) lat[i] = uint4{0, 0, 0, 0};
            if (j0 + rkey > pos_last) turned = uint4{0, 0, 0, 0};
        }
    };
    auto put_key = [&](int key, int segment, uint4 v) {
        const int ks = segment / 4, of = ks >= ks_a, in = ks - (of ? ks_a : 0);
        keys[key >> 4][of][in][16 * (segment & 3) + ((key + 4 * (in & 3)) & 15)] = v;
    };
    auto stash = [&](int c, int buf) {
        if (kg < 8) {
            // eight numbers of a key: step x / 4 of the scores, lane row x % 4
#pragma unroll
            for (int i = 0; i < 4; ++i) put_key(4 * kg + i, x, lat[i]);
            // a number without a finite size of a key that not every row sees: a weight of zero does not hide it from those that do
            // not, so it stays out of the sums, and the rows that see it lose this number at the end
            if (c * LA_CHUNK + LA_CHUNK - 1 > pos_first) {
                unsigned wild = 0;                                    // (an exponent of all ones carries into the sign's place)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const unsigned any = ((lat[i].x & 0x7f807f80u) + 0x00800080u) | ((lat[i].y & 0x7f807f80u) + 0x00800080u) |
                                         ((lat[i].z & 0x7f807f80u) + 0x00800080u) | ((lat[i].w & 0x7f807f80u) + 0x00800080u);
                    if (c * LA_CHUNK + 4 * kg + i > pos_first) wild |= any & 0x80008000u;
                }
                if (wild)
                    for (int i = 0; i < 4; ++i) {
                        const int key = c * LA_CHUNK + 4 * kg + i;
                        unsigned* pair = i == 0 ? (unsigned*)&lat[0] : i == 1 ? (unsigned*)&lat[1] : i == 2 ? (unsigned*)&lat[2] : (unsigned*)&lat[3];
                        for (int e = 0; e < 8 && key > pos_first; ++e) {
                            const unsigned half_of = e & 1 ? 0xffff0000u : 0xffffu;
                            if ((~pair[e / 2] & 0x7f807f80u & half_of) == 0) {
                                atomicMin(&lost_from[8 * x + e], key);
                                pair[e / 2] &= ~half_of;
                            }
                        }
                    }
            }
            // keys 16 kb + 4 g' + i lie at g' 8 + kb 4 + i, the order in which a lane holds their weights
            const unsigned *a = (const unsigned*)&lat[0], *b = (const unsigned*)&lat[1], *c = (const unsigned*)&lat[2], *d = (const unsigned*)&lat[3];
            const int block = x / 2, of = block >= db_a, in = block - (of ? db_a : 0);
            uint2* row = (uint2*)&Vt[buf][of][in][16 * (kg & 3)] + (kg >> 2);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const unsigned pick = e & 1 ? 0x07060302u : 0x05040100u;
                row[2 * (((x & 1) * 8 + e + 2 * (in & 3)) & 15)] =
                    uint2{__builtin_amdgcn_perm(b[e / 2], a[e / 2], pick), __builtin_amdgcn_perm(d[e / 2], c[e / 2], pick)};
            }
        }
        if (rkey < LA_CHUNK) put_key(rkey, vsteps + rx, turned);
    };
    int page_next = pt[LA_CHUNK / page_size < max_pages ? LA_CHUNK / page_size : 0];
    fetch(0, pt[0]);
    __syncthreads();                                                 // (the zeros of the keys' unused steps are there)
    stash(0, 0);
    __syncthreads();
    for (int c = 0, buf = 0; c < n_chunks; ++c, buf ^= 1) {
        if (c + 1 < n_chunks) {
            fetch(c + 1, page_next);
            if (c + 2 < n_chunks) page_next = pt[(c + 2) * LA_CHUNK / page_size];
        }
        la_f32x4 s[2], s_low[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) s[kb] = s_low[kb] = la_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KSW; ++ks) {
            const int place = 16 * g + ((n + 4 * (ks & 3)) & 15);
            const la_bf16x8 k0 = __builtin_bit_cast(la_bf16x8, keys[0][half][ks][place]);
            const la_bf16x8 k1 = __builtin_bit_cast(la_bf16x8, keys[1][half][ks][place]);
            s[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0, qh[ks], s[0], 0, 0, 0);
            s[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1, qh[ks], s[1], 0, 0, 0);
            s_low[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k0, ql[ks], s_low[0], 0, 0, 0);
            s_low[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k1, ql[ks], s_low[1], 0, 0, 0);
        }
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            s[kb] += s_low[kb];
            halves[wave][kb][lane] = s[kb];
        }
        __syncthreads();                                             // (and nobody reads this chunk's keys any more)
        // s[kb][i]: key 16 kb + 4 g + i of the chunk against row n, in powers of two
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) s[kb] += halves[wave ^ 1][kb][lane];
        if (__any(c * LA_CHUNK + LA_CHUNK - 1 > sees)) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (c * LA_CHUNK + 16 * kb + 4 * g + i > sees) s[kb][i] = -INFINITY;
        }
        float cmax = fmaxf(fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3])),
                           fmaxf(fmaxf(s[1][0], s[1][1]), fmaxf(s[1][2], s[1][3])));
        cmax = fmaxf(cmax, __shfl_xor(cmax, 16, HB_WAVE));
        cmax = fmaxf(cmax, __shfl_xor(cmax, 32, HB_WAVE));
        // (a row's sums are brought to another reference only where a weight would pass 2^LP_SLACK: by its own weights, so
        //  that nothing of it depends on the rows beside it)
        if (__any(cmax > m + LP_SLACK)) {
            const float m_new = cmax > m + LP_SLACK ? cmax : m;
            const float corr = m == m_new ? 1.0f : __builtin_amdgcn_exp2f(m - m_new);
            l *= corr;
            m = m_new;
#pragma unroll
            for (int db = 0; db < RBW; ++db)
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[db][i] *= corr;
        }
        const float base = m == -INFINITY ? 0.f : m;                 // (a row that has seen nothing yet)
        la_bf16x8 ph, pl;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float p = __builtin_amdgcn_exp2f(s[kb][i] - base);
                l += p;
                __bf16 hi, lo;
                la_split(p, hi, lo);
                ph[4 * kb + i] = hi;
                pl[4 * kb + i] = lo;
            }
#pragma unroll
        for (int db = 0; db < RBW; db += 2) {
            la_bf16x8 v[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                v[i] = __builtin_bit_cast(la_bf16x8, Vt[buf][half][db + i][16 * g + ((n + 2 * ((db + i) & 3)) & 15)]);
            }
#pragma unroll
            for (int i = 0; i < 2; ++i) acc[db + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[i], ph, acc[db + i], 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 2; ++i) acc[db + i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[i], pl, acc[db + i], 0, 0, 0);
        }
        if (c + 1 < n_chunks) stash(c + 1, buf ^ 1);
        __syncthreads();
    }
    l += __shfl_xor(l, 16, HB_WAVE);
    l += __shfl_xor(l, 32, HB_WAVE);
    if (!mine) return;
    if (sinks) l += __builtin_amdgcn_exp2f(sinks[h] * LP_LOG2E - m);                 // (an infinite share, a sink far above every score, leaves 0)
    float w = l > 0.f ? 1.0f / l : 0.f;
    if (gate) w *= 1.0f / (1.0f + expf(-gate[(size_t)t * gate_ld + h]));
#pragma unroll
    for (int db = 0; db < RBW; ++db)
        if (db < db_n) {
            // acc[db][i]: number 16 (db0 + db) + 4 g + i of row n's sum
            bf16 o[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
                o[i] = hb_from_float<bf16>(lost_from[16 * (db0 + db) + 4 * g + i] > sees ? acc[db][i] * w : NAN);
            *(uint2*)(out + ((size_t)t * H + h) * rank + 16 * (db0 + db) + 4 * g) =
                uint2{o[0].bits | ((unsigned)o[1].bits << 16), o[2].bits | ((unsigned)o[3].bits << 16)};
        }
}

// out[row, :] = sum over the ranges (in order) of their sums, brought to one maximum, over the summed
// denominators, times sigmoid(gate). One block a (token, head).
__global__ void __launch_bounds__(256)
latent_merge_kernel(const float* __restrict__ part_acc, const float* __restrict__ part_ml, bf16* __restrict__ out,
                    const float* __restrict__ gate, int gate_ld, int H, int rank, int splits,
                    const float* __restrict__ sinks) {
    __shared__ float share[HB_WAVE + 1];          // the ranges' weights, and the row's factor
    const size_t row = blockIdx.x;
    if (threadIdx.x < HB_WAVE) {
        // lane s holds range s's share (at most 64 ranges)
        const int lane = threadIdx.x;
        const bool has = lane < splits;
        const float ms = has ? part_ml[(row * splits + lane) * 2] : -INFINITY;
        const float ls = has ? part_ml[(row * splits + lane) * 2 + 1] : 0.f;
        const float m = hb_wave_max(ms);
        const float ws = ms > -INFINITY ? expf(ms - m) : 0.f;
        float l = hb_wave_sum(ls * ws);
        if (sinks) l += expf(sinks[row % H] - m);           // once, whatever the ranges
        float w = l > 0.f ? 1.0f / l : 0.f;
        if (gate) w *= 1.0f / (1.0f + expf(-gate[(row / H) * gate_ld + row % H]));
        share[lane] = ws;
        if (lane == 0) share[HB_WAVE] = w;
    }
    __syncthreads();
    const float w = share[HB_WAVE];
    const float* pa = part_acc + row * splits * rank;
    for (int d = threadIdx.x; d < rank; d += blockDim.x) {
        float a = 0.f;
        int s2 = 0;
        for (; s2 + 4 <= splits; s2 += 4) {            // (four ranges' loads at a time; summed in the ranges' order)
            const float v0 = pa[(size_t)s2 * rank + d], v1 = pa[(size_t)(s2 + 1) * rank + d];
            const float v2 = pa[(size_t)(s2 + 2) * rank + d], v3 = pa[(size_t)(s2 + 3) * rank + d];
            a = fmaf(v0, share[s2], a);
            a = fmaf(v1, share[s2 + 1], a);
            a = fmaf(v2, share[s2 + 2], a);
            a = fmaf(v3, share[s2 + 3], a);
        }
        for (; s2 < splits; ++s2) a = fmaf(pa[(size_t)s2 * rank + d], share[s2], a);
        out[row * rank + d] = hb_from_float<bf16>(a * w);
    }
}

extern "C" int hb_latent_attention_mfma(const float* q_full, const void* pages, void* out, float* part_acc,
                                        float* part_ml, const float* gate, int gate_ld, const int* positions,
                                        const int* seq_of, const int* slots, const int* page_table, int max_pages,
                                        int page_size, int T, int H, int rank, int rot, float scale, int splits,
                                        int chunks_per_split, const float* sinks, const int* seq_starts, int n_seqs,
                                        int longest, hipStream_t stream) {
    HB_REQUIRE(T > 0 && H > 0, "latent attention: empty input");
    HB_REQUIRE(rank > 0 && rank % 32 == 0 && rank <= 512 && rot % 32 == 0 && rank + rot <= 640,
               "latent attention: the matrix-core kernel takes a latent and a rotated part in steps of 32, up to 512 + 128, not %d + %d", rank, rot);
    HB_REQUIRE(page_size % LA_CHUNK == 0, "latent attention: pages of %d positions", page_size);
    HB_REQUIRE(splits >= 1 && splits <= HB_WAVE && chunks_per_split >= 1, "latent attention: %d ranges, the kernels take 1 to 64", splits);
    HB_REQUIRE(splits == 1 || (part_acc && part_ml), "latent attention: ranges need scratch");
    const long long blocks = (long long)T * ((H + 15) / 16);
    HB_REQUIRE(blocks < (1ll << 31) && (long long)T * H < (1ll << 31) - LP_ROWS, "latent attention: too many tokens for the grid");
    if (seq_starts) {      // the prompts' kernel; longest: the most tokens that a sequence of the step brings
        HB_REQUIRE(n_seqs > 0 && n_seqs <= 65535 && longest > 0 && longest <= T, "latent attention: %d sequences of up to %d tokens", n_seqs, longest);
#define LP_LAUNCH(RBV, KSV)                                                                                           \
    latent_attention_prompt_kernel<RBV, KSV>                                                                          \
        <<<dim3((unsigned)(((long long)longest * H + LP_ROWS - 1) / LP_ROWS), n_seqs), 512, 0, stream>>>(             \
            q_full, (const bf16*)pages, (bf16*)out, gate, gate_ld, positions, seq_starts, slots, page_table, max_pages, \
            page_size, H, rank, rot, scale, sinks)
        if (rank <= 128 && rank + rot <= 256) LP_LAUNCH(4, 4);
        else if (rank <= 256 && rank + rot <= 384) LP_LAUNCH(8, 6);
        else if (rank + rot <= 512) LP_LAUNCH(16, 8);
        else if (rank + rot <= 576) LP_LAUNCH(16, 9);
        else LP_LAUNCH(16, 10);
#undef LP_LAUNCH
        HB_CHECK_LAUNCH("latent_attention_prompt");
        return 0;
    }
    const dim3 grid((unsigned)blocks, splits);
#define LA_LAUNCH(RBV, KSV)                                                                                      \
    latent_attention_mfma_kernel<RBV, KSV><<<grid, HB_WAVE, 0, stream>>>(                                          \
        q_full, (const bf16*)pages, (bf16*)out, part_acc, part_ml, gate, gate_ld, positions, seq_of, slots,      \
        page_table, max_pages, page_size, H, rank, rot, scale, splits, chunks_per_split, sinks)
    if (rank <= 128 && rank + rot <= 256) LA_LAUNCH(8, 8);
    else if (rank <= 256 && rank + rot <= 384) LA_LAUNCH(16, 12);
    else LA_LAUNCH(32, 20);
#undef LA_LAUNCH
    HB_CHECK_LAUNCH("latent_attention_mfma");
    if (splits > 1) {
        latent_merge_kernel<<<(unsigned)((long long)T * H), 256, 0, stream>>>(part_acc, part_ml, (bf16*)out, gate, gate_ld, H, rank, splits, sinks);
        HB_CHECK_LAUNCH("latent_merge");
    }
    return 0;
}
