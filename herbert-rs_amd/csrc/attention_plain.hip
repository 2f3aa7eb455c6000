// Plain attention over the paged cache, float32 arithmetic, any storage types,
// any head size up to 512, any number of heads and groups.
// The keys a query at position p sees are
// [max(0, p + 1 - window), p] (window 0 = all keys from 0). They are walked in
// chunks of 64 that start at multiples of 64 of the absolute position, with an
// online softmax: the chunking, and so the rounding, depends on the positions only,
// not on how the tokens were cut into steps or batches.
// A workgroup of four waves takes 16 columns: the query heads of one key head for one token (a decode step), or for
// the next few tokens of one sequence (a prompt), each with its own mask. Both contractions run on the matrix cores in float32
// (mfma_f32.h), whose sums are chains of fmaf over ascending k: a score over the head's entries, an output over a chunk's keys. A
// wave scores 16 of a chunk's 64 keys, the scores meet in LDS, where every wave reads all 64 of its lanes' columns as the
// second product wants them (the weights never leave the registers again), and each wave owns a quarter of the
// head's entries of the output. A chunk's values are asked for before its scores are computed and the next chunk's keys after.
// The sum of a chunk's weights is a fixed tree over the keys' numbers. A chunk that a column does not see leaves
// it as it was, bit for bit, so a column's result is the same whatever tile it is in.
// Bound by a wave's instructions on a chunk (alone on its SIMD it issues one in four or five cycles): about 2.8 us a chunk of heads of 128, of which the
// products are one; 4,000 keys take 175 us, two prompts of 333 and 230 tokens, 16 heads of 128 on 8, 34 and a decode step of them 22. A
// branch an element (a weight only where there is a score, a load only within the head), every wave taking all 64 keys' exponentials, and masks and
// searches for infinities where nothing is masked cost 307, 41 and 33; two or three groups of four waves that take chunks in turn gained
// a tenth at 4,000 keys and lost up to a third of a prompt. A tile holds tokens of one sequence: a prompt of 512 tokens beside 15 single
// tokens at 4,096 keys takes 420 us, and took 2,670 where the next packed tokens were a tile whoever's they were.
// In xigh/herbert-rs: scores q . k / sqrt(hd), query head h on kv head h / (nq / nkv)
// (crates/backends/backend_common/src/generic_attention/decode.rs:126), causal by count
// (crates/backends/backend_common/src/generic_attention/prefill/kernel_f32.rs:65-67), online softmax and
// sum of p v (kernel_f32.rs:83-110; decoding: crates/backends/backend_common/src/attention_common.rs:141-178),
// all float32. The window is not in the reference, which never reads those keys. Nor is the sink: with
// `sinks` [nq] given, the softmax's denominator of head h also holds exp(sinks[h]), a score without a key
// and a value, unscaled, counted once (the running maximum starts there and the running sum at one).
// Nor are these two: with chunk > 0 the keys a query sees are those at or before it within its own chunk of
// `chunk` positions, [floor(p / chunk) chunk, p], the chunks counted from the sequence's start; with
// softcap > 0 a scaled score s becomes softcap tanh(s / softcap) before the softmax. Nor these: with `bias`
// [nq, bias_ld] given, the score of key j for query i in head h also has bias[h bias_ld + bias_at + bias_len - 1 - n]
// added (after the scale), n = min(i - j, bias_len - 1): a bias by distance, the last value from there on; and with
// keep_first > 0 (and a window) the sequence's first so many keys are seen as well.
#include "common.h"
#include "mfma_f32.h"
#include <math.h>

HB_MODULE_ERROR_SLOT()

#define HB_MAX_HEAD_DIM 512
#define CHUNK 64

// What a query row sees: keys [lo, hi) and [0, kept).
struct Seen {
    int lo, hi, kept;
};
__device__ __forceinline__ Seen seen_by(int pos, int window, int chunk, int keep_first) {
    Seen s;
    s.hi = pos + 1;
    s.lo = chunk > 0 ? pos / chunk * chunk : (window > 0 && s.hi > window) ? s.hi - window : 0;
    s.kept = keep_first < s.lo ? keep_first : s.lo;
    return s;
}

// NB: blocks of 16 of the head's entries that a wave owns of the output (the head has up to 64 NB entries). VEC: heads in
// whole quads, rows aligned, and pages that hold whole chunks. AHEAD: the next chunk's values are in flight
// while a chunk is worked on (wide heads have no registers left for that).
template <class T, class TO, int NB, bool VEC, bool AHEAD>
__global__ void __launch_bounds__(256)
attention_plain_kernel(const T* __restrict__ q, const T* __restrict__ k_cache,
                       const T* __restrict__ v_cache, TO* __restrict__ out,
                       const int* __restrict__ positions, const int* __restrict__ seq_of,
                       const int* __restrict__ slots, const int* __restrict__ page_table, int max_pages,
                       int page_size, int nq, int nkv, int hd, float scale, int window,
                       const float* __restrict__ sinks, int chunk, float softcap, const float* __restrict__ bias,
                       int bias_ld, int bias_at, int bias_len, int keep_first, int heads_a_tile,
                       const int2* __restrict__ tiles) {
    constexpr int DB = 4 * NB;                       // blocks of 16 entries of a head
    constexpr int QLD = 16 * DB + 4, SLD = CHUNK + 4;
    __shared__ __attribute__((aligned(16))) float qs[16 * QLD], ss[16 * SLD];
    __shared__ float tops[4][16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 15, g4 = lane >> 4;
    const int group = nq / nkv, tiles_a_head = (group + heads_a_tile - 1) / heads_a_tile;
    const int g = blockIdx.y / tiles_a_head, h_first = blockIdx.y % tiles_a_head * heads_a_tile;
    // (a list of the tiles' first tokens and how many they are, all of one sequence, or a token a tile)
    const int t0 = tiles ? tiles[blockIdx.x].x : blockIdx.x, n_here = tiles ? tiles[blockIdx.x].y : 1;

    // the queries, zeros beyond the head's entries and in columns that are nobody's, every 16 entries transposed
    for (int i = tid; i < 16 * 16 * DB; i += 256) {
        const int c = i / (16 * DB), d = i % (16 * DB);
        const int tok = c / heads_a_tile, head = h_first + c % heads_a_tile;
        float v = 0.f;
        if (tok < n_here && head < group && d < hd) v = hb_to_float(q[((size_t)(t0 + tok) * nq + g * group + head) * hd + d]);
        qs[c * QLD + (d & ~15) + 4 * (d & 3) + ((d >> 2) & 3)] = v;
    }
    // this lane's column
    const int my_tok = r / heads_a_tile, my_head = h_first + r % heads_a_tile;
    const bool mine = my_tok < n_here && my_head < group;
    const int h = g * group + (mine ? my_head : 0);
    const int pos = positions[t0 + (mine ? my_tok : 0)];
    const Seen see = seen_by(pos, window, chunk, keep_first);
    float m = -INFINITY, l = 0.f;
    if (sinks) m = sinks[h], l = 1.0f;
    f32x4 acc[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int* pt = page_table + (size_t)slots[seq_of[t0]] * max_pages;
    // what the tile's tokens see together
    Seen all = seen_by(positions[t0], window, chunk, keep_first);
    for (int i = 1; i < n_here; ++i) {
        const Seen s = seen_by(positions[t0 + i], window, chunk, keep_first);
        all.lo = min(all.lo, s.lo), all.hi = max(all.hi, s.hi), all.kept = max(all.kept, s.kept);
    }
    // the chunks that some token sees: those of the kept keys, then those from the window's (or the sequence's) first key on
    const int from = all.lo / CHUNK, kept_chunks = min((all.kept + CHUNK - 1) / CHUNK, from);
    const int count = kept_chunks + (all.hi + CHUNK - 1) / CHUNK - from;
    auto chunk_at = [&](int i) { return CHUNK * (i < kept_chunks ? i : from + i - kept_chunks); };
    // (keys from all.hi on are the last key once more; a table's entries are pages that exist)
    f32x4 key[DB], val[AHEAD ? NB : 1][4];
    auto fetch_keys = [&](int c, int page) {
        const int j = min(c + 16 * wave + r, all.hi - 1);
        const int in_page = VEC ? c % page_size + j - c : j % page_size;
        const T* row = k_cache + (((size_t)(VEC ? page : pt[j / page_size]) * nkv + g) * page_size + in_page) * hd;
#pragma unroll
        for (int b = 0; b < DB; ++b)
            key[b] = VEC ? load_quad<true>(row + (16 * b + 4 * g4 < hd ? 16 * b + 4 * g4 : 0), 4) : load_quad<false>(row + 16 * b + 4 * g4, hd - 16 * b - 4 * g4);
    };
    auto fetch_values = [&](int c, int page, int i, f32x4 (&to)[4]) {       // of the wave's i-th block of entries
        const T* at = v_cache + ((size_t)page * nkv + g) * hd * page_size + c % page_size + 4 * g4;
        const int d = 16 * (wave + 4 * i) + r;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            if (VEC) {      // (a page holds a whole chunk; what lies beyond all.hi is made zeros below)
                to[b] = load_quad<true>(at + (size_t)(d < hd ? d : 0) * page_size + 16 * b, 4);
                continue;
            }
            to[b] = f32x4{0.f, 0.f, 0.f, 0.f};
            const int j = c + 16 * b + 4 * g4;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (d < hd && j + e < all.hi)
                    to[b][e] = hb_to_float(v_cache[(((size_t)pt[(j + e) / page_size] * nkv + g) * hd + d) * page_size + (j + e) % page_size]);
        }
    };
    // (the page after the next is looked up a chunk before its loads are asked for; beyond the last chunk the last once more)
    auto page_at = [&](int i) { return pt[chunk_at(min(i, count - 1)) / page_size]; };
    int page = page_at(0), page_next = page_at(1);
    fetch_keys(chunk_at(0), page);
    if (AHEAD) {
#pragma unroll
        for (int i = 0; i < NB; ++i) fetch_values(chunk_at(0), page, i, val[i]);
    }
    __syncthreads();
    for (int at = 0; at < count; ++at) {
        const int c = chunk_at(at), following = chunk_at(min(at + 1, count - 1));
        if (VEC && hd < 16 * DB)
#pragma unroll
            for (int b = 0; b < DB; ++b) key[b] = 16 * b + 4 * g4 < hd ? key[b] : f32x4{0.f, 0.f, 0.f, 0.f};
        f32x4 dots = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int b = 0; b < DB; ++b) {
            transpose_quads(key[b]);
            const f32x4 qq = *(const f32x4*)&qs[r * QLD + 16 * b + 4 * g4];
#pragma unroll
            for (int s = 0; s < 4; ++s) dots = mfma_k4(key[b][s], qq[s], dots);
        }
        const int page_after = page_at(at + 2);
        if (AHEAD) fetch_keys(following, page_next);
        dots *= scale;
        if (softcap > 0.f)
#pragma unroll
            for (int e = 0; e < 4; ++e) dots[e] = softcap * tanhf(dots[e] / softcap);
        if (bias)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int n = max(0, min(pos - (c + 16 * wave + 4 * g4 + e), bias_len - 1));
                dots[e] += bias[(size_t)h * bias_ld + bias_at + bias_len - 1 - n];
            }
        const bool sees = mine && ((c < see.hi && c + CHUNK > see.lo) || c < see.kept);
        float top = -INFINITY;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int j = c + 16 * wave + 4 * g4 + e;
            dots[e] = sees && (j >= see.lo || j < see.kept) && j < see.hi ? dots[e] : -INFINITY;
            top = fmaxf(top, dots[e]);
        }
        top = fmaxf(top, __shfl_xor(top, 16, HB_WAVE));
        top = fmaxf(top, __shfl_xor(top, 32, HB_WAVE));
        if (g4 == 0) tops[wave][r] = top;
        hb_workgroup_barrier();                       // (and the weights of the chunk before have been read)
        const float m_new = fmaxf(m, fmaxf(fmaxf(tops[0][r], tops[1][r]), fmaxf(tops[2][r], tops[3][r])));
        const float corr = expf(sees ? m - m_new : 0.f);
        m = sees ? m_new : m;                         // (a chunk that is not seen does not hide a sink of NaN)
#pragma unroll
        for (int e = 0; e < 4; ++e) {                 // (the exponential in any case: no branch an element)
            const bool there = dots[e] != -INFINITY;
            const float weight = expf(there ? dots[e] - m_new : 0.f);
            ss[r * SLD + 16 * wave + 4 * e + g4] = there ? weight : 0.f;
        }
        hb_workgroup_barrier();
        // this lane's share of its column: keys 16 b + 4 s + g4
        f32x4 p[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) p[b] = *(const f32x4*)&ss[r * SLD + 16 * b + 4 * g4];
        // the tree: key j with j ^ 32, j ^ 16 (blocks), j ^ 8, j ^ 4 (quads), j ^ 2, j ^ 1 (lanes)
        f32x4 t = (p[0] + p[2]) + (p[1] + p[3]);
        float sum = (t[0] + t[2]) + (t[1] + t[3]);
        sum += __shfl_xor(sum, 32, HB_WAVE);
        sum += __shfl_xor(sum, 16, HB_WAVE);
        l = l * corr + sum;
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            acc[i] *= corr;
            f32x4 (&v)[4] = val[AHEAD ? i : 0];
            if (!AHEAD) fetch_values(c, page, i, v);
            // a value without a finite size, perhaps of a key that some column does not see: a weight of zero does
            // not hide it
            if (VEC && (c + CHUNK > all.hi || hd < 16 * DB))
#pragma unroll
                for (int b = 0; b < 4; ++b)
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[b][e] = 16 * (wave + 4 * i) + r < hd && c + 16 * b + 4 * g4 + e < all.hi ? v[b][e] : 0.f;
            f32x4 nothing = {0.f, 0.f, 0.f, 0.f};     // (or NaN)
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e) nothing[b] = fmaf(v[b][e], 0.f, nothing[b]);
            if (!__any(!((nothing[0] + nothing[1]) + (nothing[2] + nothing[3]) == 0.f))) {
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    transpose_quads(v[b]);
#pragma unroll
                    for (int s = 0; s < 4; ++s) acc[i] = mfma_k4(v[b][s], p[b][s], acc[i]);
                }
            } else {
#pragma unroll
                for (int b = 0; b < 4; ++b)
                    for (int s = 0; s < 4; ++s)
                        for (int k = 0; k < 4; ++k) {
                            const int j = c + 16 * b + 4 * s + k;
                            const float w = __shfl(s == 0 ? p[b][0] : s == 1 ? p[b][1] : s == 2 ? p[b][2] : p[b][3], 16 * k + r, HB_WAVE);
                            if (j >= all.hi) continue;
                            const T* v = v_cache + ((size_t)pt[j / page_size] * nkv + g) * hd * page_size + j % page_size;
                            const bool valid = mine && (j >= see.lo || j < see.kept) && j < see.hi;
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const int d = 16 * (wave + 4 * i) + 4 * g4 + e;
                                if (valid && d < hd) acc[i][e] = fmaf(w, hb_to_float(v[(size_t)d * page_size]), acc[i][e]);
                            }
                        }
            }
            if (AHEAD) fetch_values(following, page_next, i, v);
        }
        if (!AHEAD && at + 1 < count) fetch_keys(following, page_next);
        page = page_next, page_next = page_after;
    }
    if (!mine) return;
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    TO* row = out + ((size_t)(t0 + my_tok) * nq + h) * hd;
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int d = 16 * (wave + 4 * i) + 4 * g4 + e;
            if (d < hd) row[d] = hb_from_float<TO>(acc[i][e] * inv);
        }
}

// q, out: [T, nq * hd]; keys [pages, nkv, page_size, hd], values [pages, nkv, hd, page_size];
// dtype covers q and cache, and out unless out_dtype says float32.
// tiles [n_tiles, 2] or null: the tiles that the packed tokens are cut into, as the first token and how many, up to tokens_a_tile
// (as many as fit 16 columns beside a key head's query heads) of one sequence; null: every token is a tile.
extern "C" int hb_attention_plain(const void* q, const void* k_cache, const void* v_cache, void* out,
                                  int dtype, const int* positions, const int* seq_of, const int* slots,
                                  const int* page_table, int max_pages, int page_size, int T, const int* tiles,
                                  int n_tiles, int tokens_a_tile, int nq,
                                  int nkv, int hd, float scale, int window, const float* sinks,
                                  int chunk, float softcap, const float* bias, int bias_ld, int bias_at,
                                  int bias_len, int keep_first, int out_dtype, hipStream_t stream) {
    HB_REQUIRE(T > 0 && nq > 0 && nkv > 0, "attention: empty input");
    HB_REQUIRE(nq % nkv == 0, "attention: %d query heads not divisible by %d kv heads", nq, nkv);
    HB_REQUIRE(hd > 0 && hd <= HB_MAX_HEAD_DIM, "attention: head_dim %d not in 1..%d", hd,
               HB_MAX_HEAD_DIM);
    HB_REQUIRE(page_size > 0 && window >= 0, "attention: bad page size or window");
    HB_REQUIRE(chunk >= 0 && !(chunk > 0 && window > 0) && softcap >= 0.f, "attention: bad chunk or cap of the scores");
    HB_REQUIRE(keep_first >= 0 && (keep_first == 0 || window > 0), "attention: kept first keys go with a window");
    HB_REQUIRE(!bias || (bias_len > 0 && bias_at >= 0 && bias_at + bias_len <= bias_ld), "attention: bad table of biases");
    HB_REQUIRE(nq <= 65535, "attention: too many heads for the grid");
    HB_REQUIRE(out_dtype == dtype || out_dtype == HB_F32, "attention: the output is stored as the cache is, or in float32");
    // a key head's query heads side by side; where there is room, and a list of tiles, several tokens of a sequence
    const int group = nq / nkv, heads_a_tile = group < 16 ? group : 16;
    HB_REQUIRE(!tiles || (n_tiles > 0 && n_tiles <= T && tokens_a_tile == 16 / heads_a_tile && (uintptr_t)tiles % 8 == 0),
               "attention: a list of %d tiles of %d tokens for %d tokens and groups of %d heads", n_tiles, tokens_a_tile, T, group);
    const int tiles_a_head = (group + heads_a_tile - 1) / heads_a_tile;
    HB_REQUIRE((long long)nkv * tiles_a_head <= 65535, "attention: too many heads for the grid");
    const dim3 grid(tiles ? n_tiles : T, nkv * tiles_a_head);
    const int size = dtype == HB_F32 ? 4 : 2;
    const bool vec = hd % 4 == 0 && page_size % CHUNK == 0 && (uintptr_t)k_cache % (4 * size) == 0 && (uintptr_t)v_cache % (4 * size) == 0;
#define HB_ATTENTION(TT, TO, NB, VEC)                                                                                 \
    attention_plain_kernel<TT, TO, NB, VEC, (NB <= 2 && VEC)><<<grid, 256, 0, stream>>>(                              \
        (const TT*)q, (const TT*)k_cache, (const TT*)v_cache, (TO*)out, positions, seq_of, slots, page_table, max_pages, \
        page_size, nq, nkv, hd, scale, window, sinks, chunk, softcap, bias, bias_ld, bias_at, bias_len, keep_first,    \
        heads_a_tile, (const int2*)tiles)
#define HB_ATTENTION_OF(TT, TO)                                                                                       \
    do {                                                                                                              \
        if (!vec && hd <= 64) HB_ATTENTION(TT, TO, 1, false);                                                         \
        else if (!vec && hd <= 128) HB_ATTENTION(TT, TO, 2, false);                                                   \
        else if (!vec) HB_ATTENTION(TT, TO, 8, false);                                                                \
        else if (hd <= 64) HB_ATTENTION(TT, TO, 1, true);                                                             \
        else if (hd <= 128) HB_ATTENTION(TT, TO, 2, true);                                                            \
        else if (hd <= 256) HB_ATTENTION(TT, TO, 4, true);                                                            \
        else HB_ATTENTION(TT, TO, 8, true);                                                                           \
    } while (0)
    if (dtype == HB_BF16 && out_dtype == HB_F32) HB_ATTENTION_OF(bf16, float);
    else if (dtype == HB_F32) HB_ATTENTION_OF(float, float);
    else if (dtype == HB_BF16) HB_ATTENTION_OF(bf16, bf16);
    else HB_REQUIRE(false, "attention: unknown dtype %d", dtype);
#undef HB_ATTENTION_OF
#undef HB_ATTENTION
    HB_CHECK_LAUNCH("attention_plain");
    return 0;
}
