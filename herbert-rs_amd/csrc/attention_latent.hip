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
#include "lds_read.h"
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
// into q_full[t, h, q_at ...] (q_full [T, H, q_row] float32: rows of rank + rot, whose first `rank` are written by the
// product with W_uk^T, or of `rot` alone). One block a token.
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
                                    const float* __restrict__ q_norm_w, TC* __restrict__ c_q, int q_row, int q_at) {
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
        q_full[((size_t)t * H + h) * q_row + q_at + i] = v;
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
                               const float* q_down, int q_rank, const float* q_norm_w, void* c_q, int q_row, int q_at,
                               hipStream_t stream) {
    HB_REQUIRE(H == 0 || (q_at >= 0 && q_row >= q_at + rot), "latent write: %d turned entries at %d of rows of %d", rot, q_at, q_row);
    HB_REQUIRE(!q_down || (q_rank > 0 && q_norm_w && c_q), "latent write: a query latent needs its norm and a place");
    HB_REQUIRE(T > 0 && (H > 0 || (H == 0 && (q_down || write_cache))) && rank > 0 && rot >= 0 && qd >= 0, "latent write: empty input");
    HB_REQUIRE(rot_dims >= 0 && rot_dims <= rot && rot_dims % 2 == 0, "latent write: %d rotated of %d", rot_dims, rot);
    if (dtype == HB_F32)
        latent_write_kernel<float><<<T, 256, 0, stream>>>(down, down_ld, norm_w, q, q_ld, q_full, (bf16*)q_plain, inv_freq, positions, seq_of, slots,
                                                          page_table, max_pages, page_size, (float*)pages, H, qd,
                                                          rank, rot, rot_dims, eps, write_cache, q_down, q_rank, q_norm_w,
                                                          (float*)c_q, q_row, q_at);
    else if (dtype == HB_BF16)
        latent_write_kernel<bf16><<<T, 256, 0, stream>>>(down, down_ld, norm_w, q, q_ld, q_full, (bf16*)q_plain, inv_freq, positions, seq_of, slots,
                                                         page_table, max_pages, page_size, (bf16*)pages, H, qd,
                                                         rank, rot, rot_dims, eps, write_cache, q_down, q_rank, q_norm_w,
                                                          (bf16*)c_q, q_row, q_at);
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
// A workgroup of four waves takes 16 heads of one token (the rows of its matrix products) and a range of the keys, in
// chunks of 32; a wave takes a quarter of a row's numbers. Scores: S^T = K Q^T, the chunk's rows straight from memory as operands (a lane: one
// key's 8 consecutive numbers), the query (times the scale) in registers as two bfloat16 halves, high
// and low, so that it keeps 16 bits of mantissa (with the high half alone a test with large queries
// lost a digit). The sums are float32; the waves' parts of them meet in LDS, where every wave adds them in the waves' order. The softmax and
// its state are a lane's own (a lane holds scores of one head only) and the same in every wave. Weighted sums: O^T = V^T P^T
// with the weights again as high and low halves (they are never rounded to 8 bits), and V^T, the
// wave's part of the chunk's first `rank` numbers a key with the keys along a row, written to LDS from the registers
// that hold them as the scores' operands: it is the wave's own. A chunk's 32 keys stand there in pairs, n and 16 + n, so that a pair is one
// write and a lane's eight keys of a product one read; the weights go from the scores' registers into the product in the same order.
// The next chunk's rows are asked for as soon as a chunk's are in LDS. With more than one range a token the unnormalised sums,
// maxima and denominators go to scratch and a second kernel joins them in the ranges' order.
// Bound by its own chain: positions, slot, page, rows, scores, exchange, softmax, sums, and by code that a CU reads for the first time, which
// was four times as long by one wave that held a whole row. With the kernel that joins the ranges, by one wave | now, 16 heads of 512 + 64, us:
// 1 token at 100 keys 20.3 | 10.5, at 4,000 37 | 20; 4 at 300 22 | 12; 8 at 2,000 39 | 20; 32 at 1,000 40 | 20; 64 at 2,000 78 | 38; 200 at 300 74 | 34,
// at 1,500 209 | 88; 400 at 500 166 | 55; 128 heads, 64 at 1,000 242 | 99; 8 heads of 256 + 64, 4 at 300 13.0 | 8.3, 256 at 1,000 68 | 42.
// Sizes: rank and rot multiples of 32; VW >= rank / 128 steps of 32 numbers a wave, KX >= rot / 128 of the rotated part.
typedef __bf16 la_bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 la_bf16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 la_bf16x2 __attribute__((ext_vector_type(2)));
typedef float la_f32x4 __attribute__((ext_vector_type(4)));
#define LA_CHUNK 32
#define LA_WAVES 4
#define LA_VT_STRIDE 40          // bfloat16 a row of V^T in LDS: 32 keys and 16 bytes, so rows start at other banks

__device__ __forceinline__ void la_split(float v, __bf16& hi, __bf16& lo) {
    hi = (__bf16)v;
    lo = (__bf16)(v - (float)hi);
}

template <int VW, int KX>
__global__ void __launch_bounds__(LA_WAVES * HB_WAVE)
latent_attention_mfma_kernel(const float* __restrict__ q_full, const bf16* __restrict__ pages,
                             bf16* __restrict__ out, float* __restrict__ part_acc, float* __restrict__ part_ml,
                             const float* __restrict__ gate, int gate_ld, const int* __restrict__ positions,
                             const int* __restrict__ seq_of, const int* __restrict__ slots,
                             const int* __restrict__ page_table, int max_pages, int page_size, int H, int rank,
                             int rot, float scale, int splits, int chunks_per_split, const float* __restrict__ sinks) {
    constexpr int RB = 2 * VW, KSM = VW + KX;                // a wave's blocks of 16 sums, its steps of the scores
    __shared__ __attribute__((aligned(16))) __bf16 Vt_all[LA_WAVES][RB * 16 * LA_VT_STRIDE];
    __shared__ __attribute__((aligned(16))) la_f32x4 parts[2][LA_WAVES][2][HB_WAVE];
    const int HB = (H + 15) / 16;
    const int t = blockIdx.x / HB, hb = blockIdx.x % HB, split = blockIdx.y;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = lane & 15, g = lane >> 4;
    const int h = hb * 16 + n;
    const bool head = h < H;
    const int pos = positions[t];
    const int kd = rank + rot, KS = kd / 32, vsteps = rank / 32;
    const int v_each = (vsteps + LA_WAVES - 1) / LA_WAVES, v_first = wave * v_each;         // v_each <= VW
    const int v_mine = vsteps - v_first < v_each ? vsteps - v_first : v_each;               // (0 or less: none)
    // the wave's i-th step: of its own quarter of the latent, then every fourth of the rotated part
    auto step_at = [&](int i) { return i < VW ? v_first + i : vsteps + wave + LA_WAVES * (i - VW); };
    auto has = [&](int i) { return i < VW ? i < v_mine : step_at(i) < KS; };
    __bf16* const Vt = Vt_all[wave];
    const int n_chunks = (pos + LA_CHUNK) / LA_CHUNK;            // chunks that hold a key <= pos
    const int c_begin = split * chunks_per_split;
    const int c_end = n_chunks < c_begin + chunks_per_split ? n_chunks : c_begin + chunks_per_split;
    float m = -INFINITY, l = 0.f;
    la_f32x4 acc[RB];
#pragma unroll
    for (int db = 0; db < RB; ++db) acc[db] = la_f32x4{0.f, 0.f, 0.f, 0.f};

    if (c_begin < c_end) {
        const int* pt = page_table + (size_t)slots[seq_of[t]] * max_pages;
        la_bf16x8 qh[KSM], ql[KSM], kv[2][KSM];
        // a chunk's 32 keys lie in one page (pages hold a multiple of 32 positions)
        auto page_of = [&](int c) { return pt[(c < c_end ? c : c_end - 1) * LA_CHUNK / page_size]; };
        auto fetch = [&](int c, int page) {
            const bf16* chunk = pages + ((size_t)page * page_size + c * LA_CHUNK % page_size + n) * kd + 8 * g;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int i = 0; i < KSM; ++i)
                    if (has(i)) kv[kb][i] = *(const la_bf16x8*)(chunk + (size_t)(16 * kb) * kd + 32 * step_at(i));
        };
        const int page = page_of(c_begin);
        int page_next = page_of(c_begin + 1);
        const float* qrow = q_full + ((size_t)t * H + (head ? h : H - 1)) * kd + 8 * g;
#pragma unroll
        for (int i = 0; i < KSM; ++i)
            if (has(i)) {
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    __bf16 hi, lo;
                    la_split(qrow[32 * step_at(i) + e] * scale, hi, lo);
                    qh[i][e] = hi;
                    ql[i][e] = lo;
                }
            }
        fetch(c_begin, page);
        for (int c = c_begin; c < c_end; ++c) {
            const int j0 = c * LA_CHUNK;
            la_f32x4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int i = 0; i < KSM; ++i)
                if (has(i)) {
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb) s[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kv[kb][i], qh[i], s[kb], 0, 0, 0);
#pragma unroll
                    for (int kb = 0; kb < 2; ++kb) s[kb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kv[kb][i], ql[i], s[kb], 0, 0, 0);
                    // the same numbers are the keys' part of V^T: keys n and 16 + n, numbers 32 i + 8 g + e of the wave's
                    if (i < VW) {
#pragma unroll
                        for (int e = 0; e < 8; ++e)
                            *(la_bf16x2*)(Vt + (32 * i + 8 * g + e) * LA_VT_STRIDE + 2 * n) = la_bf16x2{kv[0][i][e], kv[1][i][e]};
                    }
                }
            if (c + 1 < c_end) {
                fetch(c + 1, page_next);
                page_next = page_of(c + 2);
            }
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) parts[c & 1][wave][kb][lane] = s[kb];
            hb_workgroup_barrier();                              // (one a chunk: the parts lie in two places by turns)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                s[kb] = parts[c & 1][0][kb][lane];
#pragma unroll
                for (int w = 1; w < LA_WAVES; ++w) s[kb] += parts[c & 1][w][kb][lane];
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
            const float m_new = fmaxf(m, cmax);                  // finite: the chunk holds a key <= pos
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
                    ph[2 * i + kb] = hi;
                    pl[2 * i + kb] = lo;
                }
            l = l * corr + psum;
            m = m_new;
#pragma unroll
            for (int db = 0; db < RB; ++db)
                if (db < 2 * v_mine) {
                    acc[db] *= corr;
                    const la_bf16x8 vv = *(const la_bf16x8*)(Vt + (db * 16 + n) * LA_VT_STRIDE + 8 * g);
                    acc[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vv, ph, acc[db], 0, 0, 0);
                    acc[db] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vv, pl, acc[db], 0, 0, 0);
                }
        }
        l += __shfl_xor(l, 16, HB_WAVE);
        l += __shfl_xor(l, 32, HB_WAVE);
    }
    if (!head) return;
    // acc[db][i]: number 32 v_first + 16 db + 4 g + i of head n's sum
    const size_t row = (size_t)t * H + h;
    const int first = 32 * v_first + 4 * g;
    if (splits == 1) {
        if (sinks) l += expf(sinks[h] - m);                 // (an infinite share, a sink far above every score, leaves 0)
        float w = l > 0.f ? 1.0f / l : 0.f;
        if (gate) w *= 1.0f / (1.0f + expf(-gate[(size_t)t * gate_ld + h]));
#pragma unroll
        for (int db = 0; db < RB; ++db)
            if (db < 2 * v_mine) {
#pragma unroll
                for (int i = 0; i < 4; ++i) out[row * rank + first + db * 16 + i] = hb_from_float<bf16>(acc[db][i] * w);
            }
    } else {
        float* pa = part_acc + (row * splits + split) * rank + first;
#pragma unroll
        for (int db = 0; db < RB; ++db)
            if (db < 2 * v_mine) *(la_f32x4*)(pa + db * 16) = acc[db];
        if (wave == 0 && g == 0) {
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
                               int rot, float scale, const float* __restrict__ sinks, const int* __restrict__ which) {
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
    const int seq = which ? which[blockIdx.y] : blockIdx.y, tile = gridDim.x - 1 - blockIdx.x;      // (the tiles with the most keys first)
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

// ------------------------------------------------ prompts with the heads' keys and values built
// Where a sequence brings many tokens, building every head's keys and values once costs less than scoring on the
// latents: a pair of query and key takes dim + rot + vdim products a head (320) in place of 2 rank + rot (1,088), and the
// two products that take queries and sums through the heads' matrices go. Two kernels: the first leaves keys and values of all
// positions that the step's sequences hold in scratch, in the order in which the second one's matrix products read them;
// so these come into LDS by plain copies and go on to the products without a bank met twice. 2,048 tokens of 16 heads, 128 + 64 and 128
// on 512: 67 us and 21 to build the heads (scoring on the latents 286, and 81 for the two products); three prompts of 1,054 to 1,400 tokens
// 87 and 38 (396 and 79).
// Scratch, in blocks of 32 keys (a sequence's tiles of 64 keys follow each other, the sequences too):
//   keys [H][block][dim / 16][64 lanes][8]: lane = key + 32 * (d / 8 % 2), the shared rotated parts [block][rot / 16][64][8] alike;
//   values [H][block][vdim / 32][2][64 lanes][8]: lane = v % 32 + 32 g, entry e of step s = key 16 s + 8 (e / 4) + 4 g + e % 4, the
//   order in which a lane of the scores' product holds its weights. Keys behind a sequence's last are zeros.
typedef float la_f32x16 __attribute__((ext_vector_type(16)));
#define LH_TILE 64
#define LH_RANK 512

// The n_seqs sequences that take this form are those that `which` names (null: all of the step, in their order). The one of them
// whose tiles hold tile `tile`, and how many tiles lie before its own.
__device__ __forceinline__ int lh_sequence_of(int tile, const int* context_lens, const int* which, int n_seqs, int& before) {
    const int lane = threadIdx.x & (HB_WAVE - 1);
    before = 0;
    for (int first = 0; first < n_seqs; first += HB_WAVE) {
        int upto = 0;
        if (first + lane < n_seqs) upto = (context_lens[which ? which[first + lane] : first + lane] + LH_TILE - 1) / LH_TILE;
#pragma unroll
        for (int off = 1; off < HB_WAVE; off <<= 1) {
            const int v = __shfl_up(upto, off, HB_WAVE);
            if (lane >= off) upto += v;
        }
        const unsigned long long beyond = __ballot(before + upto > tile);
        if (beyond) {
            const int at = __ffsll(beyond) - 1;
            if (at) before += __shfl(upto, at - 1, HB_WAVE);
            return which ? which[first + at] : first + at;
        }
        before += __shfl(upto, HB_WAVE - 1, HB_WAVE);
    }
    return -1;
}

// A workgroup: 64 keys of one head (dim = vdim); each of its four waves takes blocks of 32 of a key's and a value's numbers, one
// of either at a time. The latents come into LDS (rows 16 bytes apart beyond their length, so that 16 rows' reads spread over the banks),
// the matrices' operands straight from the L2s, a step ahead. K^T = W_uk c^T and V = c W_uv^T: what leaves is
// what a lane holds.
__global__ void __launch_bounds__(256)
latent_heads_kernel(const bf16* __restrict__ pages, const bf16* __restrict__ w_uk, const bf16* __restrict__ w_uv,
                    bf16* __restrict__ keys, bf16* __restrict__ turned, bf16* __restrict__ values,
                    const int* __restrict__ context_lens, int n_seqs, const int* __restrict__ slots,
                    const int* __restrict__ page_table, int max_pages, int page_size, int tiles, int dim, int rank,
                    int rot, const int* __restrict__ which) {
    __shared__ __attribute__((aligned(16))) char lh_lds[LH_TILE * (LH_RANK * 2 + 16)];
    const int tile = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    int before;
    const int seq = lh_sequence_of(tile, context_lens, which, n_seqs, before);
    if (seq < 0) return;
    const int key0 = (tile - before) * LH_TILE, held = context_lens[seq];
    const int kd = rank + rot, octets = rank / 8, pitch = rank * 2 + 16;
    // (a tile lies in one page)
    const bf16* row0 = pages + ((size_t)page_table[(size_t)slots[seq] * max_pages + key0 / page_size] * page_size + key0 % page_size) * kd;
    for (int i0 = tid; i0 < LH_TILE * octets; i0 += 8 * 256) {
        uint4 v[8];                                            // (eight loads on their way at a time)
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = i0 + 256 * u, key = i / octets;
            v[u] = uint4{0, 0, 0, 0};
            if (i < LH_TILE * octets && key0 + key < held) v[u] = *(const uint4*)(row0 + key * kd + 8 * (i % octets));
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = i0 + 256 * u;
            if (i < LH_TILE * octets) *(uint4*)(lh_lds + i / octets * pitch + 16 * (i % octets)) = v[u];
        }
    }
    if (h == 0)
        for (int i = tid; i < LH_TILE * (rot / 8); i += 256) {
            const int key = i / (rot / 8), o = i % (rot / 8);
            uint4 v = uint4{0, 0, 0, 0};
            if (key0 + key < held) v = *(const uint4*)(row0 + key * kd + rank + 8 * o);
            ((uint4*)turned)[(((size_t)2 * tile + key / 32) * (rot / 16) + o / 2) * HB_WAVE + key % 32 + 32 * (o & 1)] = v;
        }
    __syncthreads();
    const int n = lane & 31, g = lane >> 5, KT = rank / 32;
    const char* c_at = lh_lds + n * pitch + 16 * g;
    // operand of 32 rows x 16 k from packed blocks [k / 32][rows / 16][lane = 16 (k / 8 % 4) + row % 16][8]
    const size_t w_step = (size_t)dim / 16 * HB_WAVE * 8;
    for (int b = wave; b < dim / 32; b += 4) {
        const size_t at = (size_t)h * dim * rank + ((size_t)(2 * b + (n >> 4)) * HB_WAVE + 16 * g + (n & 15)) * 8;
        la_f32x16 kt[2], v[2];
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) kt[j][e] = v[j][e] = 0.f;
        // four steps of 32 k in flight (beyond the last: the last once more, which goes nowhere)
        la_bf16x8 wk[4][2], wv[4][2];
        auto load = [&](int to, int k) {
            const size_t kk = at + min(k, KT - 1) * w_step;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                wk[to][s] = *(const la_bf16x8*)(w_uk + kk + s * 32 * 8);
                wv[to][s] = *(const la_bf16x8*)(w_uv + kk + s * 32 * 8);
            }
        };
        auto use = [&](int from, int k) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const la_bf16x8 c = *(const la_bf16x8*)(c_at + 32 * j * pitch + 64 * k + 32 * s);
                    kt[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wk[from][s], c, kt[j], 0, 0, 0);
                    v[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(c, wv[from][s], v[j], 0, 0, 0);
                }
        };
#pragma unroll
        for (int u = 0; u < 4; ++u) load(u, u);
        int k = 0;
        for (; k + 4 <= KT; k += 4) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                __builtin_amdgcn_sched_barrier(0);
                use(u, k + u);
                load(u, k + 4 + u);
            }
        }
#pragma unroll
        for (int u = 0; u < 3; ++u)
            if (k + u < KT) use(u, k + u);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const size_t block = ((size_t)h * tiles + tile) * 2 + j;
            // kt[j][4 a + c]: number 32 b + 8 a + 4 g + c of key 32 j + n
            bf16* to = keys + (block * (dim / 16) + 2 * b) * HB_WAVE * 8;
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                bf16 o[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) o[c] = hb_from_float<bf16>(kt[j][4 * a + c]);
                *(uint2*)(to + ((a >> 1) * HB_WAVE + n + 32 * (a & 1)) * 8 + 4 * g) =
                    uint2{o[0].bits | ((unsigned)o[1].bits << 16), o[2].bits | ((unsigned)o[3].bits << 16)};
            }
            // v[j][e]: key 32 j + 8 (e / 4) + 4 g + e % 4, number 32 b + n
            to = values + (block * (dim / 32) + b) * 2 * HB_WAVE * 8;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                bf16 o[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = hb_from_float<bf16>(v[j][8 * s + e]);
                *(uint4*)(to + (s * HB_WAVE + lane) * 8) =
                    uint4{o[0].bits | ((unsigned)o[1].bits << 16), o[2].bits | ((unsigned)o[3].bits << 16),
                          o[4].bits | ((unsigned)o[5].bits << 16), o[6].bits | ((unsigned)o[7].bits << 16)};
            }
        }
    }
}

// A workgroup: 64 queries of one head and sequence, four waves: two groups of 32 queries (a lane's column) x the two blocks of a
// tile of 64 keys, so that the longest row's chain is half its keys; the two blocks' sums meet at the end. The query (times the
// scale) is two bfloat16 halves and so are the weights, as in the kernels above; the reference of the
// exponents moves as in latent_attention_prompt_kernel. A tile's keys come in while the tile before is worked on, its values while its scores
// are: two barriers a tile, 64 KB of LDS, two workgroups a CU. Bound by a tile's chain in a wave (scores, exponentials, sums: 1.7 us,
// 0.55 of it the matrix cores'), which two waves a SIMD only partly cover. The tiles with the most keys start first, those with the fewest
// follow, so that a CU that takes two of them gets one of either kind.
template <int DS, int RS, int VB>
__global__ void __launch_bounds__(256, 2)
latent_attention_heads_kernel(const float* __restrict__ q, size_t q_ld, const float* __restrict__ q_turned, int turned_ld,
                              const bf16* __restrict__ keys, const bf16* __restrict__ turned,
                              const bf16* __restrict__ values, bf16* __restrict__ out, const float* __restrict__ gate,
                              int gate_ld, const int* __restrict__ positions, const int* __restrict__ seq_starts,
                              const int* __restrict__ context_lens, int tiles, int H, float scale,
                              const float* __restrict__ sinks, const int* __restrict__ which) {
    constexpr int KS = DS + RS, DIM = 16 * DS, ROT = 16 * RS, VD = 32 * VB;
    constexpr int AHEAD = 3;                                               // reads of LDS ahead of their products
    constexpr int K_LOADS = 2 * KS / 4, V_LOADS = VB;                      // a wave's share of a tile, in kilobytes
    static_assert(2 * KS % 4 == 0, "a tile's keys are dealt out to four waves");
    __shared__ __attribute__((aligned(16))) uint4 K[2][2][KS][HB_WAVE];
    __shared__ __attribute__((aligned(16))) uint4 V[2][VB][2][HB_WAVE];
    __shared__ float met[2][2][32];                                        // the other block's reference and sum of a row
    __shared__ int lost_from[VD];                                          // [number]: the key from which on it is not finite
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 31, g = lane >> 5, group = wave & 1, block = wave >> 1;
    const int listed = blockIdx.y, seq = which ? which[listed] : listed, h = blockIdx.x % H, nth = blockIdx.x / H, most = gridDim.x / H;
    const int tile = nth < (most + 1) / 2 ? most - 1 - nth : nth - (most + 1) / 2;
    const int begin = seq_starts[seq], rows = seq_starts[seq + 1] - begin;
    if (tile * 64 >= rows) return;
    int before = 0;
    for (int s = lane; s < listed; s += HB_WAVE) before += (context_lens[which ? which[s] : s] + LH_TILE - 1) / LH_TILE;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) before += __shfl_xor(before, off, HB_WAVE);
    before = __builtin_amdgcn_readfirstlane(before);
    const int pos0 = __builtin_amdgcn_readfirstlane(positions[begin]);     // (a sequence's tokens follow each other)
    const int in_seq = tile * 64 + 32 * group + n;
    const bool mine = in_seq < rows;
    const int t = begin + (mine ? in_seq : rows - 1);
    const int sees = mine ? pos0 + in_seq : -1;
    const int first = pos0 + tile * 64;                                    // what the workgroup's first row sees
    const int last = pos0 + min(tile * 64 + 63, rows - 1);
    const int wave_last = pos0 + min(tile * 64 + 32 * group + 31, rows - 1);
    const int n_tiles = last / LH_TILE + 1;
    for (int i = tid; i < VD; i += 256) lost_from[i] = 0x7fffffff;

    const char* k_src = (const char*)(keys + ((size_t)h * tiles + before) * 2 * DS * HB_WAVE * 8) + 16 * lane;
    const char* r_src = (const char*)(turned + (size_t)before * 2 * RS * HB_WAVE * 8) + 16 * lane;
    const char* v_src = (const char*)(values + ((size_t)h * tiles + before) * 2 * VB * 2 * HB_WAVE * 8) + 16 * lane;
    auto ask_keys = [&](int c, int buf) {
#pragma unroll
        for (int i = 0; i < K_LOADS; ++i) {
            const int piece = wave * K_LOADS + i, b = piece / KS, ks = piece % KS;
            const char* src = ks < DS ? k_src + ((size_t)(2 * c + b) * DS + ks) * 1024 : r_src + ((size_t)(2 * c + b) * RS + ks - DS) * 1024;
            hb_load_to_lds(src, &K[buf][0][0][0] + piece * HB_WAVE);
        }
    };
    auto ask_values = [&](int c) {
#pragma unroll
        for (int i = 0; i < V_LOADS; ++i) {
            const int piece = wave * V_LOADS + i;
            hb_load_to_lds(v_src + ((size_t)c * 4 * VB + piece) * 1024, &V[0][0][0][0] + piece * HB_WAVE);
        }
    };
    la_bf16x8 qh[KS], ql[KS];
    {
        const float* row = q + (size_t)t * q_ld + (size_t)h * (DIM + ROT) + 8 * g;
        const float* trow = q_turned + ((size_t)t * H + h) * turned_ld + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                __bf16 hi, lo;
                la_split((ks < DS ? row[16 * ks + e] : trow[16 * (ks - DS) + e]) * (scale * LP_LOG2E), hi, lo);
                qh[ks][e] = hi;
                ql[ks][e] = lo;
            }
    }
    ask_keys(0, 0);
    float m = -INFINITY, l = 0.f;
    la_f32x16 acc[VB];
#pragma unroll
    for (int b = 0; b < VB; ++b)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[b][e] = 0.f;

    for (int c = 0, buf = 0; c < n_tiles; ++c, buf ^= 1) {
        const int key0 = c * LH_TILE + 32 * block;
        const bool works = key0 <= wave_last;
        hb_wait_vmcnt<0>();
        hb_workgroup_barrier();                      // the tile's keys are there; nobody reads the tile before any more
        ask_values(c);
        if (c + 1 < n_tiles) ask_keys(c + 1, buf ^ 1);
        la_bf16x8 ph[2], pl[2];
        if (works) {
            la_f32x16 s, s_low;
#pragma unroll
            for (int e = 0; e < 16; ++e) s[e] = s_low[e] = 0.f;
            const uint4* const at = &K[buf][block][0][lane];
            la_bf16x8 k[KS];
            static_for<0, AHEAD>([&](auto t) { k[t()] = lds_read_ahead<1024 * t()>(at); });
            static_for<0, KS>([&](auto t) {
                constexpr int ks = t();
                if constexpr (ks + AHEAD < KS) k[ks + AHEAD] = lds_read_ahead<1024 * (ks + AHEAD)>(at);
                lds_wait<(ks + AHEAD < KS ? AHEAD : KS - 1 - ks)>(k[ks]);
                s = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k[ks], qh[ks], s, 0, 0, 0);
                s_low = __builtin_amdgcn_mfma_f32_32x32x16_bf16(k[ks], ql[ks], s_low, 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            });
            s += s_low;
            // s[e]: key key0 + 8 (e / 4) + 4 g + e % 4 against query n, in powers of two
            if (__any(key0 + 31 > sees)) {
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    if (key0 + 8 * (e >> 2) + 4 * g + (e & 3) > sees) s[e] = -INFINITY;
            }
            float cmax = s[0];
#pragma unroll
            for (int e = 1; e < 16; ++e) cmax = fmaxf(cmax, s[e]);
            cmax = fmaxf(cmax, __shfl_xor(cmax, 32, HB_WAVE));
            if (__any(cmax > m + LP_SLACK)) {
                const float m_new = cmax > m + LP_SLACK ? cmax : m;
                const float corr = m == m_new ? 1.0f : __builtin_amdgcn_exp2f(m - m_new);
                l *= corr;
                m = m_new;
#pragma unroll
                for (int b = 0; b < VB; ++b)
#pragma unroll
                    for (int e = 0; e < 16; ++e) acc[b][e] *= corr;
            }
            const float base = m == -INFINITY ? 0.f : m;             // (a row that has seen nothing yet)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float p = __builtin_amdgcn_exp2f(s[e] - base);
                l += p;
                __bf16 hi, lo;
                la_split(p, hi, lo);
                ph[e >> 3][e & 7] = hi;
                pl[e >> 3][e & 7] = lo;
            }
        }
        if (c + 1 < n_tiles) hb_wait_vmcnt<K_LOADS>();               // (the values were asked for before the next keys)
        else hb_wait_vmcnt<0>();
        hb_workgroup_barrier();
        if (c * LH_TILE + LH_TILE - 1 > first) {
            // Keys that not every row sees: a weight of zero does not hide a number without a finite size from the rows that
            // do not see it, so such a number stays out of the sums, and the rows that see its key lose it at the end.
            for (int i = tid; i < 2 * VB * 2 * HB_WAVE; i += 256) {
                uint4* at = &V[0][0][0][0] + i;
                const uint4 v = *at;
                const unsigned any = (((v.x & 0x7f807f80u) + 0x00800080u) | ((v.y & 0x7f807f80u) + 0x00800080u) |
                                      ((v.z & 0x7f807f80u) + 0x00800080u) | ((v.w & 0x7f807f80u) + 0x00800080u)) & 0x80008000u;
                if (any) {
                    const int b = i / (VB * 2 * HB_WAVE), step = i / HB_WAVE % 2, of = i % HB_WAVE;
                    const int number = 32 * (i / (2 * HB_WAVE) % VB) + of % 32;
                    unsigned short* entry = (unsigned short*)at;
                    for (int e = 0; e < 8; ++e) {
                        const int key = c * LH_TILE + 32 * b + 16 * step + 8 * (e >> 2) + 4 * (of >> 5) + (e & 3);
                        if (key > first && (entry[e] & 0x7f80) == 0x7f80) {
                            atomicMin(&lost_from[number], key);
                            entry[e] = 0;
                        }
                    }
                }
            }
            hb_workgroup_barrier();
        }
        if (works) {
            const uint4* const at = &V[block][0][0][lane];
            la_bf16x8 v[2 * VB];
            static_for<0, AHEAD>([&](auto t) { v[t()] = lds_read_ahead<1024 * t()>(at); });
            static_for<0, 2 * VB>([&](auto t) {
                constexpr int i = t(), b = i / 2, s = i % 2;
                if constexpr (i + AHEAD < 2 * VB) v[i + AHEAD] = lds_read_ahead<1024 * (i + AHEAD)>(at);
                lds_wait<(i + AHEAD < 2 * VB ? AHEAD : 2 * VB - 1 - i)>(v[i]);
                acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v[i], ph[s], acc[b], 0, 0, 0);
                acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v[i], pl[s], acc[b], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            });
        }
    }
    l += __shfl_xor(l, 32, HB_WAVE);
    __syncthreads();
    // the second block's sums go through the keys' place
    static_assert(sizeof(K) >= 2 * VB * 16 * HB_WAVE * sizeof(float), "the sums of two waves fit where the keys lay");
    float* there = (float*)&K[0][0][0][0] + group * VB * 16 * HB_WAVE + lane;
    if (block == 1) {
#pragma unroll
        for (int b = 0; b < VB; ++b)
#pragma unroll
            for (int e = 0; e < 16; ++e) there[(b * 16 + e) * HB_WAVE] = acc[b][e];
        if (g == 0) met[group][0][n] = m, met[group][1][n] = l;
    }
    __syncthreads();
    if (block == 1 || !mine) return;
    const float m1 = met[group][0][n], top = fmaxf(m, m1);
    const float base = top == -INFINITY ? 0.f : top;
    const float f0 = __builtin_amdgcn_exp2f(m - base), f1 = __builtin_amdgcn_exp2f(m1 - base);
    l = l * f0 + met[group][1][n] * f1;
    if (sinks) l += __builtin_amdgcn_exp2f(sinks[h] * LP_LOG2E - base);    // (an infinite share, a sink far above every score, leaves 0)
    float w = l > 0.f ? 1.0f / l : 0.f;
    if (gate) w *= 1.0f / (1.0f + expf(-gate[(size_t)t * gate_ld + h]));
    const float w0 = f0 * w, w1 = f1 * w;
    bf16* to = out + ((size_t)t * H + h) * VD + 4 * g;
#pragma unroll
    for (int b = 0; b < VB; ++b)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            // acc[b][4 a + e]: number 32 b + 8 a + 4 g + e of query n
            bf16 o[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float v = acc[b][4 * a + e] * w0 + there[(b * 16 + 4 * a + e) * HB_WAVE] * w1;
                o[e] = hb_from_float<bf16>(lost_from[32 * b + 8 * a + 4 * g + e] > sees ? v : NAN);
            }
            *(uint2*)(to + 32 * b + 8 * a) = uint2{o[0].bits | ((unsigned)o[1].bits << 16), o[2].bits | ((unsigned)o[3].bits << 16)};
        }
}

// tiles: the tiles of 64 keys of the sequences together that `which` names (n_seqs of the step's; null: its first n_seqs), longest: the most
// tokens that one of them brings; scratch: keys [H][2 tiles][dim / 16][64][8], turned [2 tiles][rot / 16][64][8], values [H][2 tiles][vdim / 32]
// [2][64][8]. q_turned: the queries' rotated parts, turned_ld floats from a head's to the next. w_uk / w_uv: [H] matrices of dim / vdim rows of
// rank, packed. Other sequences' rows of out are left as they are.
extern "C" int hb_latent_attention_heads(const float* q, int q_ld, const float* q_turned, int turned_ld, const void* pages, const void* w_uk,
                                         const void* w_uv, void* keys, void* turned, void* values, void* out,
                                         const float* gate, int gate_ld, const int* positions, const int* seq_starts,
                                         const int* context_lens, int n_seqs, const int* slots, const int* page_table,
                                         int max_pages, int page_size, int tiles, int longest, int T, int H, int dim,
                                         int vdim, int rank, int rot, float scale, const float* sinks, const int* which,
                                         hipStream_t stream) {
    HB_REQUIRE(T > 0 && H > 0 && H <= 65535 && n_seqs > 0 && n_seqs <= 65535 && longest > 0 && longest <= T,
               "latent attention: %d sequences of up to %d of %d tokens, %d heads", n_seqs, longest, T, H);
    HB_REQUIRE(turned_ld >= rot, "latent attention: rotated parts of %d in rows of %d", rot, turned_ld);
    HB_REQUIRE(rank > 0 && rank % 32 == 0 && rank <= LH_RANK, "latent attention: built heads take a latent in steps of 32 up to 512, not %d", rank);
    HB_REQUIRE((dim == 64 || dim == 128) && vdim == dim && (rot == 0 || rot == 32 || rot == 64),
               "latent attention: heads of %d + %d and %d are not built", dim, rot, vdim);
    HB_REQUIRE(page_size > 0 && page_size % LH_TILE == 0, "latent attention: pages of %d positions", page_size);
    HB_REQUIRE(tiles > 0 && q_ld >= H * (dim + rot), "latent attention: empty input");
    const long long blocks = ((long long)longest + 63) / 64 * H;
    HB_REQUIRE(blocks < (1ll << 23) && tiles < (1 << 23), "latent attention: too many tokens for the grid");
    latent_heads_kernel<<<dim3(tiles, H), 256, 0, stream>>>((const bf16*)pages, (const bf16*)w_uk, (const bf16*)w_uv, (bf16*)keys, (bf16*)turned,
                                                            (bf16*)values, context_lens, n_seqs, slots, page_table, max_pages, page_size,
                                                            tiles, dim, rank, rot, which);
    HB_CHECK_LAUNCH("latent_heads");
    const dim3 grid((unsigned)blocks, n_seqs);
#define LH_LAUNCH(DSV, RSV, VBV)                                                                                    \
    latent_attention_heads_kernel<DSV, RSV, VBV><<<grid, 256, 0, stream>>>(                                         \
        q, (size_t)q_ld, q_turned, turned_ld, (const bf16*)keys, (const bf16*)turned, (const bf16*)values, (bf16*)out, gate, gate_ld, \
        positions, seq_starts, context_lens, tiles, H, scale, sinks, which)
    if (dim == 128) {
        if (rot == 64) LH_LAUNCH(8, 4, 4);
        else if (rot == 32) LH_LAUNCH(8, 2, 4);
        else LH_LAUNCH(8, 0, 4);
    } else {
        if (rot == 64) LH_LAUNCH(4, 4, 2);
        else if (rot == 32) LH_LAUNCH(4, 2, 2);
        else LH_LAUNCH(4, 0, 2);
    }
#undef LH_LAUNCH
    HB_CHECK_LAUNCH("latent_attention_heads");
    return 0;
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
                                        int longest, const int* which, hipStream_t stream) {
    HB_REQUIRE(T > 0 && H > 0, "latent attention: empty input");
    HB_REQUIRE(rank > 0 && rank % 32 == 0 && rank <= 512 && rot >= 0 && rot % 32 == 0 && rot <= 128,
               "latent attention: the matrix-core kernel takes a latent and a rotated part in steps of 32, up to 512 + 128, not %d + %d", rank, rot);
    HB_REQUIRE(page_size % LA_CHUNK == 0, "latent attention: pages of %d positions", page_size);
    HB_REQUIRE(splits >= 1 && splits <= HB_WAVE && chunks_per_split >= 1, "latent attention: %d ranges, the kernels take 1 to 64", splits);
    HB_REQUIRE(splits == 1 || (part_acc && part_ml), "latent attention: ranges need scratch");
    const long long blocks = (long long)T * ((H + 15) / 16);
    HB_REQUIRE(blocks < (1ll << 31) && (long long)T * H < (1ll << 31) - LP_ROWS, "latent attention: too many tokens for the grid");
    // the prompts' kernel, for the n_seqs sequences that `which` names (null: all of the step); longest: the most tokens that one brings
    if (seq_starts) {
        HB_REQUIRE(n_seqs > 0 && n_seqs <= 65535 && longest > 0 && longest <= T, "latent attention: %d sequences of up to %d tokens", n_seqs, longest);
#define LP_LAUNCH(RBV, KSV)                                                                                           \
    latent_attention_prompt_kernel<RBV, KSV>                                                                          \
        <<<dim3((unsigned)(((long long)longest * H + LP_ROWS - 1) / LP_ROWS), n_seqs), 512, 0, stream>>>(             \
            q_full, (const bf16*)pages, (bf16*)out, gate, gate_ld, positions, seq_starts, slots, page_table, max_pages, \
            page_size, H, rank, rot, scale, sinks, which)
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
#define LA_LAUNCH(VWV, KXV)                                                                                      \
    latent_attention_mfma_kernel<VWV, KXV><<<grid, LA_WAVES * HB_WAVE, 0, stream>>>(                               \
        q_full, (const bf16*)pages, (bf16*)out, part_acc, part_ml, gate, gate_ld, positions, seq_of, slots,      \
        page_table, max_pages, page_size, H, rank, rot, scale, splits, chunks_per_split, sinks)
    if (rank <= 128) LA_LAUNCH(1, 1);
    else if (rank <= 256) LA_LAUNCH(2, 1);
    else LA_LAUNCH(4, 1);
#undef LA_LAUNCH
    HB_CHECK_LAUNCH("latent_attention_mfma");
    if (splits > 1) {
        latent_merge_kernel<<<(unsigned)((long long)T * H), 256, 0, stream>>>(part_acc, part_ml, (bf16*)out, gate, gate_ld, H, rank, splits, sinks);
        HB_CHECK_LAUNCH("latent_merge");
    }
    return 0;
}
