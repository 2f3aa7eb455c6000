// A feed-forward of many small experts of which each token uses a few.
//   route     the router's logits (+ bias) of a token -> its `top` experts (largest logits, the
//             lower index of equals), weighed by exp(logit) normalised over those experts alone
//   group     the (token, choice) pairs in the order of their experts, so that an expert's rows
//             are consecutive, and a list of row tiles (expert, first row, rows) of fixed length
//   products  a tile's rows times its expert's matrix, float32 sums over k ascending by one
//             thread each (plain), whatever else is in the batch
//   activate  g = min(gate, limit), u = clamp(up, -limit, limit): y = g sigmoid(alpha g) (u + shift)
//             (limit infinite, alpha 1, shift 0: silu(gate) up)
//   combine   a token's rows weighted and summed in the order of its choices, added to the output
// Nothing here asks the host: the grids depend on the step's size only, so a step can be recorded
// and replayed.
#include "common.h"
#include "mfma_split.h"
#include <math.h>

HB_MODULE_ERROR_SLOT()

#define MOE_TILE_M 64
#define MOE_TILE_N 64
#define MOE_TILE_K 16
#define MOE_MAX_E_PER_LANE 16

// ------------------------------------------------------------------------ route
// Two ways to choose. By logits (by_scores 0): the largest logits (+ bias), weights a softmax over the chosen. By scores
// s = sigmoid(logit): the choice runs on s + correction, the weights on s itself:
// the experts form n_groups equal runs of adjacent experts, a group is worth the two highest of its
// selection values, added; only the experts of the `keep` best groups can be chosen (the lower index of equals,
// for groups as for experts), and the chosen experts' scores are divided by their sum + 1e-20.
// Three parameters change the form: softmax_scores (s is the softmax of the logits over all E experts instead of
// their sigmoids), worth_top (how many of a group's highest selection values make its worth: 2, or 1), renorm
// (0: the weights are the chosen experts' scores as they are).
struct RouteForm {
    int by_scores, n_groups, keep, softmax_scores, worth_top, renorm;
};

// The largest of a wave's 64 numbers, in every lane.
__device__ __forceinline__ unsigned wave_max_u32(unsigned v) {
#define HB_STEP(CTRL, ROWS)                                                                      \
    {                                                                                            \
        const unsigned o = (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false); \
        v = v > o ? v : o;                                                                       \
    }
    HB_STEP(0x111, 0xf) HB_STEP(0x112, 0xf) HB_STEP(0x114, 0xf) HB_STEP(0x118, 0xf)   // along the rows of 16
    HB_STEP(0x142, 0xa) HB_STEP(0x143, 0xc)                                           // a row's last lane to the next, two rows' to the others
#undef HB_STEP
    return (unsigned)__builtin_amdgcn_readlane((int)v, HB_WAVE - 1);
}

// The choice of one token by one wave: lane l holds experts l, l + 64, ... A selection value becomes a number that sorts
// as it does (0: not to be chosen, 1: not a number), the largest of the wave's goes through the lanes' neighbours instead
// of the LDS, and who holds it is a mask of lanes: some 150 clocks a chosen expert. Every wave of the workgroup calls it
// together; a and b (E and n_groups floats) are the wave's own LDS, used only where there are groups.
template <int PER>
__device__ __forceinline__ void route_token(const float* __restrict__ logits, const float* __restrict__ bias, const RouteForm f,
                                            int E, int top, float* a, float* b, int* chosen, int* chosen_too, float* weight,
                                            bool stores) {
    const int lane = threadIdx.x % HB_WAVE;
    float c[PER], s[PER];                                // selection values and scores
    unsigned key[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int e = lane + HB_WAVE * i;
        s[i] = e < E ? logits[e] : -INFINITY;
        c[i] = bias && e < E ? bias[e] : 0.f;
    }
    if (f.by_scores) {
        float top_logit = -INFINITY, denom = 1.0f;
        if (f.softmax_scores) {
#pragma unroll
            for (int i = 0; i < PER; ++i) top_logit = fmaxf(top_logit, s[i]);
            top_logit = hb_wave_max(top_logit);
            float part = 0.f;
#pragma unroll
            for (int i = 0; i < PER; ++i)
                if (lane + HB_WAVE * i < E) part += expf(s[i] - top_logit);
            denom = hb_wave_sum(part);
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) s[i] = f.softmax_scores ? expf(s[i] - top_logit) / denom : 1.0f / (1.0f + expf(-s[i]));
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        c[i] += s[i];
        const unsigned u = __float_as_uint(c[i] + 0.f);  // (-0 sorts as 0)
        const bool live = lane + HB_WAVE * i < E && !(f.by_scores && c[i] == -INFINITY);
        key[i] = !live ? 0u : c[i] != c[i] ? 1u : (u >> 31) ? ~u : u | 0x80000000u;
    }
    if (f.by_scores && f.n_groups > 1) {
        const int size = E / f.n_groups;
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (lane + HB_WAVE * i < E) a[lane + HB_WAVE * i] = c[i];
        __syncthreads();
        for (int g = lane; g < f.n_groups; g += HB_WAVE) {
            float x = -INFINITY, y = -INFINITY;          // the largest and the second
            for (int i = 0; i < size; ++i) {
                const float v = a[g * size + i];
                y = v > x ? x : v > y ? v : y;
                x = v > x ? v : x;
            }
            b[g] = (size > 1 && f.worth_top > 1) ? x + y : x;
        }
        __syncthreads();
        for (int g = lane; g < f.n_groups; g += HB_WAVE) {
            int ahead = 0;
            for (int o = 0; o < f.n_groups; ++o) ahead += (b[o] > b[g] || (b[o] == b[g] && o < g)) ? 1 : 0;
            a[g] = ahead < f.keep ? 1.f : 0.f;           // (the values have been read: a group's worth needs no more of them)
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < PER; ++i)
            if (lane + HB_WAVE * i < E && a[(lane + HB_WAVE * i) / size] == 0.f) key[i] = 0u;
    }
    float first = 0.f, sum = 0.f;
    for (int j = 0; j < top; ++j) {
        unsigned mine = key[0];
#pragma unroll
        for (int i = 1; i < PER; ++i) mine = mine > key[i] ? mine : key[i];
        const unsigned best = wave_max_u32(mine);
        int at = 0;                                      // (none left: only where the host's checks or infinite corrections allow it)
        float value = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s[0]), 0));
        bool found = best == 0u;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const unsigned long long who = __ballot(key[i] == best);
            if (!found && who) {
                const int l = __ffsll((long long)who) - 1;
                found = true;
                at = HB_WAVE * i + l;
                value = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(f.by_scores ? s[i] : c[i]), l));
                if (lane == l) key[i] = 0u;
            }
        }
        if (!f.by_scores) {
            if (j == 0) first = value;                   // the first choice is the largest
            value = expf(value - first);
        }
        sum += value;
        if (stores && lane == j % HB_WAVE) {             // (the lane that divides it below)
            chosen[j] = at;
            if (chosen_too) chosen_too[j] = at;
            weight[j] = value;
        }
    }
    if (!stores || (f.by_scores && !f.renorm)) return;
    const float total = f.by_scores ? sum + 1e-20f : sum;
    for (int j = lane; j < top; j += HB_WAVE) weight[j] /= total;
}

template <int PER>
__global__ void __launch_bounds__(HB_WAVE)
moe_route_kernel(const float* __restrict__ logits, int ld, const float* __restrict__ bias, int* __restrict__ chosen,
                 float* __restrict__ weight, int E, int top, RouteForm form) {
    __shared__ float a[HB_WAVE * PER], b[HB_WAVE * PER];
    const size_t t = blockIdx.x;
    route_token<PER>(logits + t * ld, bias, form, E, top, a, b, chosen + t * top, nullptr, weight + t * top, true);
}

// ------------------------------------------------------------------------ group
// Block e < E: the pairs of expert e, in the order of the pairs, to rows [first, first + count) and
// the expert's tiles into the list; block E: the list's unused end. order[row] = pair,
// row_of[pair] = row. Every block counts all experts' pairs for itself (a histogram in LDS), so that
// no kernel has to run before it. Experts from `real` on have no matrices (their output is their input): their
// pairs get rows like any others, but their tiles are marked as holding nothing, so no product runs on them.
// Each of the 16 waves goes over a run of the pairs of its own, twice: counting, then placing behind the waves before it
// (two barriers in all). Choice and placing of 2,048 tokens, 8 of 64 experts: 64 us with a workgroup of four waves that met
// at three barriers every 256 pairs, and a choice through the LDS; 12 now.
__global__ void __launch_bounds__(1024)
moe_place_kernel(const int* __restrict__ chosen, int* __restrict__ counts, int* __restrict__ order,
                 int* __restrict__ row_of, int* __restrict__ tile_expert, int* __restrict__ tile_row0,
                 int* __restrict__ tile_rows, int A, int E, int max_tiles, int real, int* __restrict__ tall,
                 int tall_m, int max_tall, int top, int shared_rows) {
    __shared__ int hist[HB_WAVE * MOE_MAX_E_PER_LANE];
    __shared__ int wave_n[16], firsts[16], tiles[16], talls[16];
    const int e = blockIdx.x;
    const int lane = threadIdx.x & (HB_WAVE - 1), wave = threadIdx.x / HB_WAVE;
    const int run = ((A + 1023) / 1024) * HB_WAVE;       // pairs of a wave
    const int a0 = min(A, wave * run), a1 = min(A, a0 + run);
    for (int i = threadIdx.x; i < E; i += 1024) hist[i] = 0;
    __syncthreads();
    int hits = 0;
    for (int at = a0; at < a1; at += 4 * HB_WAVE) {
        int x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = at + i * HB_WAVE + lane < a1 ? chosen[at + i * HB_WAVE + lane] : -1;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (x[i] >= 0) atomicAdd(&hist[x[i]], 1);
            hits += __popcll(__ballot(x[i] == e));
        }
    }
    if (lane == 0) wave_n[wave] = hits;
    __syncthreads();
    const int before = (int)threadIdx.x < min(e, E) ? hist[threadIdx.x] : 0;       // (E is at most the workgroup's threads)
    int first = before, tile0 = (before + MOE_TILE_M - 1) / MOE_TILE_M, tall0 = tall_m ? (before + tall_m - 1) / tall_m : 0;
#pragma unroll
    for (int off = HB_WAVE / 2; off > 0; off >>= 1) {
        first += __shfl_xor(first, off, HB_WAVE);
        tile0 += __shfl_xor(tile0, off, HB_WAVE);
        tall0 += __shfl_xor(tall0, off, HB_WAVE);
    }
    if (lane == 0) {
        firsts[wave] = first;
        tiles[wave] = tile0;
        talls[wave] = tall0;
    }
    __syncthreads();
    first = tile0 = tall0 = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
        first += firsts[w];
        tile0 += tiles[w];
        tall0 += talls[w];
    }
    if (e == E) {
        // (behind all pairs a row a token for the expert that every token takes, the matrices after the others')
        for (int t = threadIdx.x; t < shared_rows; t += 1024) order[A + t] = t * top;
        for (int i = threadIdx.x; tile0 + i < max_tiles; i += 1024) {
            const int left = shared_rows - i * MOE_TILE_M;
            tile_expert[tile0 + i] = left > 0 ? real : -1;
            if (left > 0) tile_row0[tile0 + i] = A + i * MOE_TILE_M, tile_rows[tile0 + i] = min(left, MOE_TILE_M);
        }
        for (int i = threadIdx.x; tall_m && tall0 + i < max_tall; i += 1024) {
            const int left = shared_rows - i * tall_m;
            tall[tall0 + i] = left > 0 ? real : -1;
            if (left > 0) tall[max_tall + tall0 + i] = A + i * tall_m, tall[2 * max_tall + tall0 + i] = min(left, tall_m);
        }
        return;
    }
    const int count = hist[e];
    if (threadIdx.x == 0) counts[e] = count;
    for (int i = threadIdx.x; i * MOE_TILE_M < count; i += 1024) {
        tile_expert[tile0 + i] = e < real ? e : -1;
        tile_row0[tile0 + i] = first + i * MOE_TILE_M;
        tile_rows[tile0 + i] = count - i * MOE_TILE_M < MOE_TILE_M ? count - i * MOE_TILE_M : MOE_TILE_M;
    }
    for (int i = threadIdx.x; tall_m && i * tall_m < count; i += 1024) {
        tall[tall0 + i] = e < real ? e : -1;
        tall[max_tall + tall0 + i] = first + i * tall_m;
        tall[2 * max_tall + tall0 + i] = count - i * tall_m < tall_m ? count - i * tall_m : tall_m;
    }
    if (hits == 0) return;
    int row = first;
    for (int w = 0; w < wave; ++w) row += wave_n[w];
    for (int at = a0; at < a1; at += 4 * HB_WAVE) {
        int x[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = at + i * HB_WAVE + lane < a1 ? chosen[at + i * HB_WAVE + lane] : -1;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const unsigned long long mask = __ballot(x[i] == e);
            if (x[i] == e) {
                const int pair = at + i * HB_WAVE + lane, r = row + __popcll(mask & ((1ull << lane) - 1ull));
                order[r] = pair;
                row_of[pair] = r;
            }
            row += __popcll(mask);
        }
    }
}

// Both of a step of few tokens (decode) in one launch of one workgroup, a wave a token: the choices stay in LDS, a thread
// a pair counts the pairs of its expert before it. Bound by its own chain of latencies: 8 of 64 experts for one token
// 4.4 us, for 8 tokens 5.9 (16 and 17 by the two kernels before; 16 tokens 8.1, which the two kernels now do in 6.7: the
// line lies at 8 tokens).
#define FEW_TOKENS 8
#define FEW_PAIRS 128
template <int PER>
__global__ void __launch_bounds__(HB_WAVE * FEW_TOKENS)
moe_route_few_kernel(const float* __restrict__ logits, int ld, const float* __restrict__ bias, int* __restrict__ chosen,
                     float* __restrict__ weight, int* __restrict__ counts, int* __restrict__ order, int* __restrict__ row_of,
                     int* __restrict__ tile_expert, int* __restrict__ tile_row0, int* __restrict__ tile_rows, int T, int E,
                     int top, int max_tiles, int real, int shared_rows, RouteForm form) {
    __shared__ float a[FEW_TOKENS][HB_WAVE * PER], b[FEW_TOKENS][HB_WAVE * PER];
    __shared__ __attribute__((aligned(16))) int pair_expert[FEW_PAIRS + 4];
    __shared__ int hist[HB_WAVE * PER];
    __shared__ unsigned start[HB_WAVE * PER + 1];        // an expert's first tile (upper half) and row (lower half)
    const int lane = threadIdx.x & (HB_WAVE - 1), wave = threadIdx.x / HB_WAVE;
    const int A = T * top, threads = blockDim.x;
    for (int i = threadIdx.x; i < HB_WAVE * PER; i += threads) hist[i] = 0;
    const size_t t = min(wave, T - 1);
    route_token<PER>(logits + t * ld, bias, form, E, top, a[wave], b[wave], chosen + t * top, pair_expert + t * top,
                     weight + t * top, wave < T);
    __syncthreads();
    for (int p = threadIdx.x; p < A; p += threads) atomicAdd(&hist[pair_expert[p]], 1);
    __syncthreads();
    if (wave == 0) {                                     // PER experts a lane
        unsigned own[PER], sum = 0;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int n = hist[lane * PER + i];
            own[i] = sum;
            sum += ((unsigned)((n + MOE_TILE_M - 1) / MOE_TILE_M) << 16) | (unsigned)n;
        }
        unsigned upto = sum;
#pragma unroll
        for (int off = 1; off < HB_WAVE; off <<= 1) {
            const unsigned o = __shfl_up(upto, off, HB_WAVE);
            if (lane >= off) upto += o;
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) start[lane * PER + i] = upto - sum + own[i];
        if (lane == HB_WAVE - 1) start[HB_WAVE * PER] = upto;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += threads) {
        const int n = hist[e], tile0 = start[e] >> 16, row0 = start[e] & 0xffff;
        counts[e] = n;
        for (int i = 0; i * MOE_TILE_M < n; ++i) {
            tile_expert[tile0 + i] = e < real ? e : -1;
            tile_row0[tile0 + i] = row0 + i * MOE_TILE_M;
            tile_rows[tile0 + i] = min(n - i * MOE_TILE_M, MOE_TILE_M);
        }
    }
    const int used = start[HB_WAVE * PER] >> 16;
    for (int i = used + threadIdx.x; i < max_tiles; i += threads) {
        const bool own = i == used && shared_rows > 0;     // (the expert that every token takes: up to FEW_TOKENS rows)
        tile_expert[i] = own ? real : -1;
        if (own) tile_row0[i] = A, tile_rows[i] = shared_rows;
    }
    if ((int)threadIdx.x < shared_rows) order[A + threadIdx.x] = threadIdx.x * top;
    for (int p = threadIdx.x; p < A; p += threads) {
        const int e = pair_expert[p];
        int r = start[e] & 0xffff;
        for (int q = 0; q < p; q += 4) {
            const int4 v = *(const int4*)(pair_expert + q);
            r += (v.x == e) + (v.y == e && q + 1 < p) + (v.z == e && q + 2 < p) + (v.w == e && q + 3 < p);
        }
        order[r] = p;
        row_of[p] = r;
    }
}

// tall [3, max_tall] (or null): the same list for tiles of tall_m rows, an expert, a first row and the rows of each.
// shared_rows T (or 0): after the pairs' rows, and after their tiles in either list, come a row a token of one more expert, number
// `real`, that every token takes: order there is token times top.
// logits' rows are ld floats apart (their first E count).
// by_scores 0: the largest logits (+ bias), weights a softmax over the chosen.
// by_scores 1: sigmoid scores, `bias` is the correction of the choice, n_groups groups of which `keep` count.
extern "C" int hb_moe_route(const float* logits, const float* bias, int* chosen, float* weight, int* counts,
                            int* order, int* row_of, int* tile_expert, int* tile_row0, int* tile_rows, int T, int E,
                            int top, int max_tiles, int ld, int by_scores, int n_groups, int keep, int real,
                            int softmax_scores, int worth_top, int renorm, int* tall, int tall_m, int max_tall,
                            int shared_rows, hipStream_t stream) {
    HB_REQUIRE(tall_m == 0 || ((tall_m == 128 || tall_m == 192 || tall_m == 256) && tall), "moe: row tiles of %d", tall_m);
    HB_REQUIRE(ld >= E, "moe: logits rows %d apart for %d experts", ld, E);
    HB_REQUIRE(!by_scores || (n_groups > 0 && E % n_groups == 0 && keep > 0 && keep <= n_groups &&
                              top <= keep * (E / n_groups)),
               "moe: %d of %d groups of %d experts cannot give %d experts", keep, n_groups, E, top);
    HB_REQUIRE(T > 0 && E > 0 && top > 0 && top <= E, "moe: %d of %d experts for %d tokens", top, E, T);
    HB_REQUIRE(real > 0 && real <= E, "moe: %d of %d experts have matrices", real, E);
    HB_REQUIRE(E <= HB_WAVE * MOE_MAX_E_PER_LANE, "moe: %d experts, the router takes up to %d", E, HB_WAVE * MOE_MAX_E_PER_LANE);
    const long long A = (long long)T * top;
    HB_REQUIRE(A < (1ll << 30), "moe: too many (token, expert) pairs");
    HB_REQUIRE(shared_rows == 0 || (shared_rows == T && real == E), "moe: %d rows of a shared expert for %d tokens, %d of %d experts with matrices",
               shared_rows, T, real, E);
    HB_REQUIRE(max_tiles >= (A + MOE_TILE_M - 1) / MOE_TILE_M + E + (shared_rows + MOE_TILE_M - 1) / MOE_TILE_M &&
                   (tall_m == 0 || max_tall >= (A + tall_m - 1) / tall_m + E + (shared_rows + tall_m - 1) / tall_m),
               "moe: the tile list is too short");
    const RouteForm form = {by_scores, n_groups, keep, softmax_scores, worth_top, renorm};
    if (T <= FEW_TOKENS && A <= FEW_PAIRS && E <= HB_WAVE * 4 && tall_m == 0) {
#define HB_FEW(PER)                                                                                                      \
    moe_route_few_kernel<PER><<<1, HB_WAVE * (T < 4 ? 4 : T), 0, stream>>>(logits, ld, bias, chosen, weight, counts, order, \
        row_of, tile_expert, tile_row0, tile_rows, T, E, top, max_tiles, real, shared_rows, form)
        if (E <= HB_WAVE) HB_FEW(1);
        else if (E <= HB_WAVE * 2) HB_FEW(2);
        else HB_FEW(4);
#undef HB_FEW
        HB_CHECK_LAUNCH("moe_route_few");
        return 0;
    }
#define HB_ROUTE(PER) moe_route_kernel<PER><<<T, HB_WAVE, 0, stream>>>(logits, ld, bias, chosen, weight, E, top, form)
    if (E <= HB_WAVE) HB_ROUTE(1);
    else if (E <= HB_WAVE * 2) HB_ROUTE(2);
    else if (E <= HB_WAVE * 4) HB_ROUTE(4);
    else HB_ROUTE(MOE_MAX_E_PER_LANE);
#undef HB_ROUTE
    HB_CHECK_LAUNCH("moe_route");
    moe_place_kernel<<<E + 1, 1024, 0, stream>>>(chosen, counts, order, row_of, tile_expert, tile_row0, tile_rows, (int)A, E, max_tiles, real, tall, tall_m, max_tall,
                                              top, shared_rows);
    HB_CHECK_LAUNCH("moe_place");
    return 0;
}

// ------------------------------------------------------------------------ products, plain
// C[row, n] = sum_k A[src(row), k] * W[e][n, k] for the rows of every tile; src(row) = order[row] / top
// (the token's row of the activations) if `top` > 0, else the row itself.
template <class TA, class TW, class TC>
__global__ void __launch_bounds__(256)
moe_gemm_plain_kernel(const TA* __restrict__ A, const TW* __restrict__ W, TC* __restrict__ C,
                      const int* __restrict__ order, const int* __restrict__ tile_expert,
                      const int* __restrict__ tile_row0, const int* __restrict__ tile_rows, int top, int N, int K) {
    __shared__ float As[MOE_TILE_K][MOE_TILE_M + 1];
    __shared__ float Ws[MOE_TILE_K][MOE_TILE_N + 1];
    __shared__ int src[MOE_TILE_M];
    const int e = tile_expert[blockIdx.y];
    if (e < 0) return;
    const int row0 = tile_row0[blockIdx.y], rows = tile_rows[blockIdx.y];
    const int tid = threadIdx.x;
    const int tx = tid % 16, ty = tid / 16;
    const int n0 = blockIdx.x * MOE_TILE_N;
    const TW* We = W + (size_t)e * N * K;
    if (tid < MOE_TILE_M) src[tid] = tid < rows ? (top > 0 ? order[row0 + tid] / top : row0 + tid) : -1;
    __syncthreads();

    float acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = 0.f;

    for (int k0 = 0; k0 < K; k0 += MOE_TILE_K) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int el = tid + i * 256;
            const int kk = el % MOE_TILE_K, rr = el / MOE_TILE_K;
            const int k = k0 + kk, n = n0 + rr;
            As[kk][rr] = (src[rr] >= 0 && k < K) ? hb_to_float(A[(size_t)src[rr] * K + k]) : 0.f;
            Ws[kk][rr] = (n < N && k < K) ? hb_to_float(We[(size_t)n * K + k]) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < MOE_TILE_K; ++kk) {
            float a[4], w[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = As[kk][ty + 16 * i];
#pragma unroll
            for (int j = 0; j < 4; ++j) w[j] = Ws[kk][tx + 16 * j];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = fmaf(a[i], w[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = ty + 16 * i;
        if (r >= rows) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int n = n0 + tx + 16 * j;
            if (n < N) C[(size_t)(row0 + r) * N + n] = hb_from_float<TC>(acc[i][j]);
        }
    }
}

// The same where rows lie on 16-byte borders: the split products of mfma_split.h, a workgroup on 32 rows of an expert's matrix and all of a
// tile's rows, a wave on every stretch of k (up to GROUPED_WAVES at a time), the stretches' sums added in their order. Up to 16
// rows are one pass over the matrix' rows and bound by their bytes, more rows two blocks of 16 at a time, which read them again from
// the caches. Gate and up of two tokens, four of 8 experts each (1536 x 2048), 24 us, their down product (2048 x 768) 15; of 200 tokens, four of
// 32 experts each, 155 and 85; the kernel above, one chain of vector multiply-adds: 268, 101, 462 and 155.
#define GROUPED_WAVES 8
template <class TA, class TW, int MB, int AHEAD, int A_AHEAD>
__device__ __forceinline__ void grouped_plain_rows(const TA* __restrict__ A, const TW* __restrict__ We, float* __restrict__ C, const int* src, int from,
                                                   int rows, int row0, int n0, int N, int K, f32x4* sums) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const int r = lane & 15, q = lane >> 4;
    constexpr int NB = 2;
    const TW* w_row[NB];
    const TA* a_row[MB];
#pragma unroll
    for (int j = 0; j < NB; ++j) w_row[j] = We + (size_t)(n0 + 16 * j + r < N ? n0 + 16 * j + r : n0) * K;
#pragma unroll
    for (int i = 0; i < MB; ++i) a_row[i] = A + (size_t)src[from + 16 * i + r < rows ? from + 16 * i + r : 0] * K;
    f32x4 total[NB][MB];
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int i = 0; i < MB; ++i) total[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int first = 0; first < K; first += waves * SPLIT_STRETCH) {
        f32x4 top[NB][MB], low[NB][MB];
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int i = 0; i < MB; ++i) top[j][i] = low[j][i] = f32x4{0.f, 0.f, 0.f, 0.f};
        sum_stretch<AHEAD, A_AHEAD>(w_row, a_row, first + wave * SPLIT_STRETCH, K, q, top, low);
        __syncthreads();                              // (the sums before have been read)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int i = 0; i < MB; ++i) sums[((wave * NB + j) * MB + i) * HB_WAVE + lane] = top[j][i] + low[j][i];
        __syncthreads();
        if (wave == 0)
            for (int b = 0; b < waves && first + b * SPLIT_STRETCH < K; ++b)
#pragma unroll
                for (int j = 0; j < NB; ++j)
#pragma unroll
                    for (int i = 0; i < MB; ++i) total[j][i] += sums[((b * NB + j) * MB + i) * HB_WAVE + lane];
    }
    if (wave) return;
    mend_blocks<TA, TW>([=](int i) { return from + i < rows ? A + (size_t)src[from + i] * K : nullptr; }, We, K, n0, N, K, SPLIT_STRETCH, total);
#pragma unroll
    for (int i = 0; i < MB; ++i) {
        const int m = from + 16 * i + r;
        if (m >= rows) continue;
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int n = n0 + 16 * j + 4 * q + e;
                if (n < N) C[(size_t)(row0 + m) * N + n] = total[j][i][e];
            }
    }
}

template <class TA, class TW>
__global__ void __launch_bounds__(GROUPED_WAVES * HB_WAVE, 2)
moe_gemm_split_kernel(const TA* __restrict__ A, const TW* __restrict__ W, float* __restrict__ C, const int* __restrict__ order,
                      const int* __restrict__ tile_expert, const int* __restrict__ tile_row0, const int* __restrict__ tile_rows,
                      int top, int N, int K) {
    __shared__ int src[MOE_TILE_M];
    __shared__ f32x4 sums[GROUPED_WAVES * 4 * HB_WAVE];
    const int e = tile_expert[blockIdx.y];
    if (e < 0) return;
    const int row0 = tile_row0[blockIdx.y], rows = tile_rows[blockIdx.y], n0 = blockIdx.x * 32;
    if (threadIdx.x < MOE_TILE_M) src[threadIdx.x] = (int)threadIdx.x < rows ? (top > 0 ? order[row0 + threadIdx.x] / top : row0 + (int)threadIdx.x) : 0;
    __syncthreads();
    const TW* We = W + (size_t)e * N * K;
    if (rows <= 16)
        grouped_plain_rows<TA, TW, 1, 8, 8>(A, We, C, src, 0, rows, row0, n0, N, K, sums);
    else
        for (int from = 0; from < rows; from += 32) {
            grouped_plain_rows<TA, TW, 2, 4, 4>(A, We, C, src, from, rows, row0, n0, N, K, sums);
            __syncthreads();
        }
}

// A [rows, K] (the tokens' rows if top > 0, else one row a pair), W [E, N, K], C [pairs, N].
extern "C" int hb_moe_gemm_plain(const void* A, int a_dtype, const void* W, int w_dtype, void* C, int c_dtype,
                                 const int* order, const int* tile_expert, const int* tile_row0,
                                 const int* tile_rows, int max_tiles, int top, int N, int K, hipStream_t stream) {
    HB_REQUIRE(N > 0 && K > 0 && max_tiles > 0 && max_tiles <= 65535 * 16, "moe product: empty or too large");
    HB_REQUIRE(max_tiles <= 65535, "moe product: %d row tiles exceed the grid", max_tiles);
    const dim3 grid((N + MOE_TILE_N - 1) / MOE_TILE_N, max_tiles);
    const int key = a_dtype * 4 + w_dtype * 2 + c_dtype;
    const int stretches = (K + SPLIT_STRETCH - 1) / SPLIT_STRETCH, waves = stretches < GROUPED_WAVES ? stretches : GROUPED_WAVES;
    const bool split = K % (a_dtype == HB_F32 && w_dtype == HB_F32 ? 4 : 8) == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0;
#define HB_MOE(TA, TW, TC)                                                                                        \
    if (split)                                                                                                    \
        moe_gemm_split_kernel<TA, TW><<<dim3((N + 31) / 32, max_tiles), HB_WAVE * waves, 0, stream>>>(            \
            (const TA*)A, (const TW*)W, (float*)C, order, tile_expert, tile_row0, tile_rows, top, N, K);          \
    else                                                                                                          \
        moe_gemm_plain_kernel<TA, TW, TC><<<grid, 256, 0, stream>>>((const TA*)A, (const TW*)W, (TC*)C, order,    \
                                                                    tile_expert, tile_row0, tile_rows, top, N, K)
    switch (key) {
        case 0: HB_MOE(float, float, float); break;
        case 2: HB_MOE(float, bf16, float); break;
        case 4: HB_MOE(bf16, float, float); break;
        case 6: HB_MOE(bf16, bf16, float); break;
        default: HB_REQUIRE(false, "moe product: dtypes (%d, %d, %d) are not built (the sums are float32)", a_dtype, w_dtype, c_dtype);
    }
#undef HB_MOE
    HB_CHECK_LAUNCH("moe_gemm_plain");
    return 0;
}

// ------------------------------------------------------------------------ activate
// gu [pairs, 2 F] float32 (gate columns, then up columns) -> act [pairs, F]
template <class TOut>
__global__ void moe_activate_kernel(const float* __restrict__ gu, TOut* __restrict__ act, int F, size_t total,
                                    float limit, float alpha, float shift) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const size_t r = i / F;
        const int n = (int)(i % F);
        const float g = fminf(gu[r * 2 * F + n], limit);
        const float u = fminf(fmaxf(gu[r * 2 * F + F + n], -limit), limit);
        act[i] = hb_from_float<TOut>(g / (1.0f + expf(-alpha * g)) * (u + shift));
    }
}

extern "C" int hb_moe_activate(const float* gu, void* act, int act_dtype, int rows, int F, float limit, float alpha,
                               float shift, hipStream_t stream) {
    HB_REQUIRE(rows > 0 && F > 0, "moe activation: empty input");
    const size_t total = (size_t)rows * F;
    const size_t blocks = (total + 255) / 256;
    const unsigned grid = (unsigned)(blocks > 8192 ? 8192 : blocks);
    if (act_dtype == HB_F32)
        moe_activate_kernel<float><<<grid, 256, 0, stream>>>(gu, (float*)act, F, total, limit, alpha, shift);
    else if (act_dtype == HB_BF16)
        moe_activate_kernel<bf16><<<grid, 256, 0, stream>>>(gu, (bf16*)act, F, total, limit, alpha, shift);
    else
        HB_REQUIRE(false, "moe activation: unknown output dtype %d", act_dtype);
    HB_CHECK_LAUNCH("moe_activate");
    return 0;
}

// ------------------------------------------------------------------------ combine
// x[t, :] += sum_j weight[t, j] * y[row_of[t * top + j], :]    (float32, j ascending)
// shared [T, H] (or null): a part that every token takes, added times sigmoid(gate[t * gate_ld]).
// input [T, H] (or null) with chosen [T, top] and real: a pair whose expert is `real` or beyond has no row in y;
// its output is the token's own input row.
// A thread takes PER neighbouring columns of a token (four where rows lie in whole quads), so that a step of few tokens is
// one round of loads: 4 tokens of 2,048 columns, four rows each 4 us, 2,048 tokens 18 (a column a thread and a row's
// columns eight after another: 15 and 32).
template <int PER>
struct alignas(4 * PER) MoeColumns {
    float v[PER];
};
template <int PER>
__device__ __forceinline__ MoeColumns<PER> moe_columns(const float* p) {
    return *(const MoeColumns<PER>*)p;
}
template <int PER>
__device__ __forceinline__ MoeColumns<PER> moe_columns(const bf16* p) {
    struct alignas(2 * PER) Stored {
        bf16 v[PER];
    };
    const Stored s = *(const Stored*)p;
    MoeColumns<PER> c;
#pragma unroll
    for (int i = 0; i < PER; ++i) c.v[i] = hb_to_float(s.v[i]);
    return c;
}

struct Combined {
    const float *y, *weight;
    const int* row_of;
    int top, H;
    const float *shared, *gate;
    int gate_ld;
    const void* input;
    const int* chosen;
    int real;
};
// Columns at .. at + PER - 1 of token t: what x holds and the weighted sum.
template <class TIn, int PER>
__device__ __forceinline__ MoeColumns<PER> moe_combined(const Combined& c, const float* x, int t, int at, float open) {
    MoeColumns<PER> sum = moe_columns<PER>(x);
    for (int j0 = 0; j0 < c.top; j0 += 8) {
        MoeColumns<PER> rows[8];
        float w[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (j0 + j < c.top) {
                const size_t pair = (size_t)t * c.top + j0 + j;
                w[j] = c.weight[pair];
                if (c.input != nullptr && c.chosen[pair] >= c.real)
                    rows[j] = moe_columns<PER>((const TIn*)c.input + (size_t)t * c.H + at);
                else
                    rows[j] = moe_columns<PER>(c.y + (size_t)c.row_of[pair] * c.H + at);
            }
        MoeColumns<PER> s = {};
#pragma unroll
        for (int j = 0; j < 8; ++j)
            if (j0 + j < c.top) {
#pragma unroll
                for (int i = 0; i < PER; ++i) s.v[i] = fmaf(w[j], rows[j].v[i], s.v[i]);
            }
        if (c.shared && j0 == 0) {
            const MoeColumns<PER> part = moe_columns<PER>(c.shared + (size_t)t * c.H + at);
#pragma unroll
            for (int i = 0; i < PER; ++i) s.v[i] = fmaf(open, part.v[i], s.v[i]);
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) sum.v[i] += s.v[i];
    }
    return sum;
}

template <class TIn, int PER>
__global__ void moe_combine_kernel(Combined c, float* __restrict__ x) {
    const int t = blockIdx.x, at = (blockIdx.y * blockDim.x + threadIdx.x) * PER;
    if (at >= c.H) return;
    const float open = c.shared ? 1.0f / (1.0f + expf(-c.gate[(size_t)t * c.gate_ld])) : 0.f;
    float* out = x + (size_t)t * c.H + at;
    *(MoeColumns<PER>*)out = moe_combined<TIn, PER>(c, out, t, at, open);
}

// The same where a norm of the whole row follows (a block whose norm comes after the sum): acc holds what the sum is added to,
// x <- sum / rms(sum) * w, y <- x in its own type, acc <- alpha_next x (alpha_next 0: acc stays). A workgroup a token, four
// columns a thread and PASS, the row in registers between its sum of squares and the stores. For the few tokens of a decode
// step, where either kernel is a chain of loads and a turn between two launches. Four experts and a shared one, us in one | in two,
// 2,048 columns: 1 token 3.2 | 5.9, 8 tokens 3.4 | 5.8, 64 3.5 | 5.9, 128 3.7 | 6.1, 512 6.1 | 9.2; 4,096 columns: 8 tokens 4.5 | 7.1, 64 4.7 | 7.5, 512 12.4 | 17.7.
template <class TOut, int PASSES>
__global__ void __launch_bounds__(512)
moe_combine_norm_kernel(Combined c, float* __restrict__ acc, const float* __restrict__ w, float eps, float* __restrict__ x,
                        TOut* __restrict__ y, float alpha_next) {
    __shared__ float red[16];
    const int t = blockIdx.x;
    const float open = c.shared ? 1.0f / (1.0f + expf(-c.gate[(size_t)t * c.gate_ld])) : 0.f;
    MoeColumns<4> sum[PASSES];
    float4 weight[PASSES];
    float ss = 0.f;
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
        const int at = (p * blockDim.x + threadIdx.x) * 4;
        sum[p] = {}, weight[p] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (at >= c.H) continue;
        weight[p] = *(const float4*)(w + at);
        sum[p] = moe_combined<float, 4>(c, acc + (size_t)t * c.H + at, t, at, open);
#pragma unroll
        for (int i = 0; i < 4; ++i) ss = fmaf(sum[p].v[i], sum[p].v[i], ss);
    }
    ss = hb_block_sum(ss, red);
    const float inv = 1.0f / sqrtf(ss / (float)c.H + eps);
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
        const int at = (p * blockDim.x + threadIdx.x) * 4;
        if (at >= c.H) continue;
        const float by[4] = {weight[p].x, weight[p].y, weight[p].z, weight[p].w};
        MoeColumns<4> o, next;
        struct alignas(4 * sizeof(TOut)) {
            TOut v[4];
        } stored;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            o.v[i] = sum[p].v[i] * inv * by[i];
            next.v[i] = alpha_next * o.v[i];
            stored.v[i] = hb_from_float<TOut>(o.v[i]);
        }
        const size_t place = (size_t)t * c.H + at;
        *(MoeColumns<4>*)(x + place) = o;
        if (y) *(decltype(stored)*)(y + place) = stored;
        if (alpha_next != 0.f) *(MoeColumns<4>*)(acc + place) = next;
    }
}

extern "C" int hb_moe_combine(const float* y, const float* weight, const int* row_of, float* x, int T, int top, int H,
                              const float* shared, const float* gate, int gate_ld, const void* input,
                              int input_dtype, const int* chosen, int real, hipStream_t stream) {
    HB_REQUIRE(shared == nullptr || (gate != nullptr && gate_ld > 0), "moe combine: a shared part needs its gate");
    HB_REQUIRE(T > 0 && top > 0 && H > 0, "moe combine: empty input");
    HB_REQUIRE(input == nullptr || chosen != nullptr, "moe combine: experts without matrices need the choices");
    const bool quads = H % 4 == 0 && (uintptr_t)y % 16 == 0 && (uintptr_t)x % 16 == 0 && (uintptr_t)shared % 16 == 0 &&
                       (uintptr_t)input % 16 == 0;
    const int threads = H >= 1024 ? 256 : 64, per = quads ? 4 : 1;
    const dim3 grid(T, (H + threads * per - 1) / (threads * per));
    HB_REQUIRE(grid.y <= 65535, "moe combine: rows of %d columns exceed the grid", H);
#define HB_COMBINE(TIn, PER)                                                                                          \
    moe_combine_kernel<TIn, PER><<<grid, threads, 0, stream>>>(                                                       \
        Combined{y, weight, row_of, top, H, shared, gate, gate_ld, input, chosen, real}, x)
    const bool narrow = input != nullptr && input_dtype == HB_BF16;
    if (quads && narrow) HB_COMBINE(bf16, 4);
    else if (quads) HB_COMBINE(float, 4);
    else if (narrow) HB_COMBINE(bf16, 1);
    else HB_COMBINE(float, 1);
#undef HB_COMBINE
    HB_CHECK_LAUNCH("moe_combine");
    return 0;
}

// acc [T, H] holds what the sums are added to; see moe_combine_norm_kernel. H in steps of 4 up to 8192, rows on 16-byte borders.
extern "C" int hb_moe_combine_norm(const float* y, const float* weight, const int* row_of, float* acc, int T, int top, int H,
                                   const float* shared, const float* gate, int gate_ld, const float* norm_w, float eps, float* x,
                                   void* rows, int rows_dtype, float alpha_next, hipStream_t stream) {
    HB_REQUIRE(shared == nullptr || (gate != nullptr && gate_ld > 0), "moe combine: a shared part needs its gate");
    HB_REQUIRE(T > 0 && top > 0 && H > 0 && H % 4 == 0 && H <= 8192, "moe combine: rows of %d columns", H);
    HB_REQUIRE(((uintptr_t)y | (uintptr_t)acc | (uintptr_t)shared | (uintptr_t)norm_w | (uintptr_t)x | (uintptr_t)rows) % 16 == 0,
               "moe combine: rows off 16-byte borders");
    HB_REQUIRE(rows_dtype == HB_F32 || rows_dtype == HB_BF16, "moe combine: unknown output dtype %d", rows_dtype);
    const Combined c{y, weight, row_of, top, H, shared, gate, gate_ld, nullptr, nullptr, 0};
    const int quads = H / 4, threads = quads <= 512 ? (quads + HB_WAVE - 1) / HB_WAVE * HB_WAVE : 512;
#define HB_COMBINE(TOut, PASSES) moe_combine_norm_kernel<TOut, PASSES><<<T, threads, 0, stream>>>(c, acc, norm_w, eps, x, (TOut*)rows, alpha_next)
#define HB_COMBINE_TO(TOut)                      \
    do {                                         \
        if (quads <= 512) HB_COMBINE(TOut, 1);   \
        else if (quads <= 1024) HB_COMBINE(TOut, 2); \
        else HB_COMBINE(TOut, 4);                \
    } while (0)
    if (rows_dtype == HB_F32) HB_COMBINE_TO(float);
    else HB_COMBINE_TO(bf16);
#undef HB_COMBINE_TO
#undef HB_COMBINE
    HB_CHECK_LAUNCH("moe_combine_norm");
    return 0;
}

// ------------------------------------------------------------------------ products on the matrix cores
// The same products for bfloat16 operands with float32 sums (v_mfma_f32_16x16x32_bf16), and more
// generally a group of products that share a shape: group g multiplies rows of A (from column
// g * a_group_off on) with its own matrix W[g] [N, K] into columns of C from g * c_group_off on.
// W[g] is stored in the order of the operands, [K / 32][N / 16][64 lanes][8] (the 1 KB of 16 rows and 32 k
// in a row, lane = 16 (k / 8 % 4) + n % 16): a wave's load is one contiguous KB, where rows K apart
// would each give 64 bytes from addresses a power of two apart.
// The rows of a group come as a list of tiles (group, first row, rows <= 64) or, without a list, as
// every group's ceil(M / 64) tiles of the same M rows (heads that each have a matrix of their own).
// A workgroup is four waves on one tile of 64 rows; a wave holds four blocks of 16 weight rows
// against up to four blocks of 16 activation rows (the blocks beyond the tile's rows are skipped, so
// a tile of a few rows costs little more than streaming its weights). The weights go from memory
// straight into the lanes (lane l of an operand holds 8 consecutive k of row l % 16 from k0 + 8 (l / 16)),
// a stage ahead of their products; the tile's activations, which the four waves share, through two
// stages in LDS.
// An output is summed over k in the same order whatever else the tile holds.
// 2,048 tokens, 4 of 32 experts of 768 on 2,048: gate/up 104 us (496 TFLOP/s), down 71; a product a head of 2,048 rows, 16
// heads, 512 x 128 22 us. (With every block of columns of a tile on another XCD, so that each L2 fetched all weights for
// itself, and sums stored one by one: 141, 96 and 45. Tiles of 128 rows, one wave a SIMD: 141 and 118; two stages of weights in flight
// beside the one multiplied, or no branch around the blocks of rows that a tile lacks: no faster.)
// EPI 0: float32 C. EPI 1: bfloat16 C. EPI 2: W[g] is [2 F, K], gate rows then up rows; a wave's two
// blocks are 16 gate rows and the 16 up rows that go with them, and C [*, F] bfloat16 receives
// min(gate, limit) sigmoid(alpha min(gate, limit)) (clamp(up, -limit, limit) + shift).
typedef __bf16 hb_bf16x8 __attribute__((ext_vector_type(8)));
typedef float hb_f32x4 __attribute__((ext_vector_type(4)));

#define XCDS 8
#define TILE_RUN 4            // tiles that follow each other on an XCD
#define GM_KSTEP 64           // k a stage of the activations' ring in LDS

template <int EPI>
__global__ void __launch_bounds__(256)
grouped_mfma_kernel(const bf16* __restrict__ A, int lda, size_t a_group_off, const bf16* __restrict__ W, int N,
                    int K, void* __restrict__ Cv, int ldc, size_t c_group_off, const int* __restrict__ order,
                    int top, const int* __restrict__ tile_group, const int* __restrict__ tile_row0,
                    const int* __restrict__ tile_rows, int M, int m_tiles, float limit, float alpha, float shift, int tiles,
                    int columns, int quads) {
    // the tile's activations, a stage of 64 k at a time, as 16-byte pieces [k piece][row]: a wave's operand
    // (16 rows of one piece) is 256 contiguous bytes
    __shared__ __attribute__((aligned(16))) hb_bf16x8 a_lds[2][GM_KSTEP / 8][MOE_TILE_M];
    // Workgroups go to the XCDs in turn. TILE_RUN neighbouring tiles of a block of columns, mostly one group's, which read the
    // same weights, are given to one XCD one after another; such runs are dealt out, the blocks of columns of a run side by side.
    const int turn = blockIdx.x / XCDS, run = turn / TILE_RUN * XCDS + blockIdx.x % XCDS;
    const int tile = run / columns * TILE_RUN + turn % TILE_RUN, column = run % columns;
    if (tile >= tiles) return;
    int group, row0, rows;
    if (tile_group) {
        group = tile_group[tile];
        if (group < 0) return;
        row0 = tile_row0[tile];
        rows = tile_rows[tile];
    } else {
        group = tile / m_tiles;
        row0 = (tile % m_tiles) * MOE_TILE_M;
        rows = M - row0 < MOE_TILE_M ? M - row0 : MOE_TILE_M;
    }
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int r16 = lane & 15, g4 = lane >> 4;
    const int F = N / 2;
    const int out_cols = EPI == 2 ? F : N;
    // the wave's output columns: 64 of them, or with EPI 2 32 (from 32 gate rows and the 32 up rows that go with them)
    const int n0 = EPI == 2 ? (column * 4 + wave) * 32 : (column * 4 + wave) * 64;
    const bool idle = n0 >= out_cols;            // (such a wave still helps to load the activations)
    // W[g] lies in the operands' order [K / 32][N / 16][64 lanes][8]: a block of 16 rows and 32 k is 1 KB in a row
    const bf16* Wg = W + (size_t)group * N * K;
    const size_t kstep = (size_t)(N / 16) * 512;         // from a block to the same rows' next 32 k
    const bf16* wrow[4];
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        int nb = (EPI == 2 ? (a < 2 ? n0 + 16 * a : F + n0 + 16 * (a - 2)) : n0 + 16 * a) / 16;
        if (nb >= N / 16 || idle) nb = N / 16 - 1;       // (read a block that exists; its sums are not stored)
        wrow[a] = Wg + (size_t)nb * 512 + lane * 8;
    }
    const int blocks = (rows + 15) / 16;
    // what this thread brings of a stage: rows tid / 8 and 32 + tid / 8, piece tid % 8
    const bf16* asrc[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        int m = 32 * j + tid / 8;
        if (m >= rows) m = rows - 1;
        const int src = top > 0 ? order[row0 + m] / top : row0 + m;
        asrc[j] = A + (size_t)src * lda + (size_t)group * a_group_off + (tid % 8) * 8;
    }
    hb_f32x4 acc[4][4];
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = hb_f32x4{0.f, 0.f, 0.f, 0.f};

    const int stages = (K + GM_KSTEP - 1) / GM_KSTEP;
    hb_bf16x8 areg[2], wnext[2][4];
    auto fetch = [&](int st) {
        const int k0 = st * GM_KSTEP;
        const bool tail = k0 + (tid % 8) * 8 >= K;          // (K in steps of 32: the last stage may be half)
#pragma unroll
        for (int j = 0; j < 2; ++j) areg[j] = tail ? hb_bf16x8{} : *(const hb_bf16x8*)(asrc[j] + k0);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int a = 0; a < 4; ++a)
                wnext[h][a] = k0 + 32 * h < K ? *(const hb_bf16x8*)(wrow[a] + (size_t)(k0 / 32 + h) * kstep) : hb_bf16x8{};
    };
    fetch(0);
    for (int st = 0; st < stages; ++st) {
        const int buf = st & 1;
#pragma unroll
        for (int j = 0; j < 2; ++j) a_lds[buf][tid % 8][32 * j + tid / 8] = areg[j];
        hb_bf16x8 wv[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int a = 0; a < 4; ++a) wv[h][a] = wnext[h][a];
        __syncthreads();          // the stage is in LDS (and the stage before the last has been read by all)
        if (st + 1 < stages) fetch(st + 1);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            hb_bf16x8 xv[4];
#pragma unroll
            for (int b = 0; b < 4; ++b)
                if (b < blocks) xv[b] = a_lds[buf][4 * h + g4][16 * b + r16];
#pragma unroll
            for (int b = 0; b < 4; ++b)
                if (b < blocks) {
#pragma unroll
                    for (int a = 0; a < 4; ++a)
                        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[h][a], xv[b], acc[a][b], 0, 0, 0);
                }
        }
    }
    if (idle) return;
    // lane: activation row b * 16 + r16, weight rows g4 * 4 + i of each block
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const int m = b * 16 + r16;
        if (b >= blocks || m >= rows) continue;
        const size_t base = (size_t)(row0 + m) * ldc + (size_t)group * c_group_off;
        // (four neighbouring columns a lane: N, and with EPI 2 F, are whole blocks of 16)
#pragma unroll
        for (int a = 0; a < (EPI == 2 ? 2 : 4); ++a) {
            const int n = n0 + 16 * a + g4 * 4;
            if (n >= out_cols) continue;
            hb_f32x4 v = acc[a][b];
            if (EPI == 2) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float g = fminf(acc[a][b][i], limit);
                    const float u = fminf(fmaxf(acc[a + 2][b][i], -limit), limit);
                    v[i] = g / (1.0f + expf(-alpha * g)) * (u + shift);
                }
            }
            bf16 o[4];
            if (EPI != 0) {
#pragma unroll
                for (int i = 0; i < 4; ++i) o[i] = hb_from_float<bf16>(v[i]);
            }
            if (!quads) {                                   // (rows of C that start anywhere)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (EPI == 0) ((float*)Cv)[base + n + i] = v[i];
                    else ((bf16*)Cv)[base + n + i] = o[i];
                }
            } else if (EPI == 0) {
                *(hb_f32x4*)((float*)Cv + base + n) = v;
            } else {
                *(uint2*)((bf16*)Cv + base + n) = uint2{o[0].bits | ((unsigned)o[1].bits << 16), o[2].bits | ((unsigned)o[3].bits << 16)};
            }
        }
    }
}

// The same for groups of many rows: a workgroup on 32 TM rows (128, 192 or 256) and 256 weight rows (EPI 2: 128 gate rows and the
// 128 up rows that go with them, in turns of 16), each of four waves on 128 weight rows x 16 TM rows. What bounds
// it are the bytes that a CU takes out of the caches, 48 to 64 KB a step of 64 k here, which last
// longer than the step's products, so the tile is as high as a group's rows fill it (rows beyond a tile's own read its last row
// again, which costs no such bytes). The kernel above reads the weights for every 64 rows. Weights and activations go straight into rings in LDS (hb_load_to_lds),
// waited for by count before a bare barrier. There is no branch in the main loop; reads and loads are dealt
// out between the products, the reads of a k-step during the products of the one before. The weights' third stage lets their loads, two
// steps ahead, go out during a step's first 32 k and the activations' during its second, so that a CU's loads last the whole step. An
// activation row is 128 bytes, its 16-byte
// chunk c at chunk c ^ ((row >> 1) & 7); a block of 16 weight rows and 32 k is 1 KB as packed. K in steps of 64.
// Gate/up of 32 experts of 768 on 2,048, weights from memory (40 us at the rate of a large copy), by tiles of 64 and by the tile that
// tall_rows of moe.py takes, in brackets that one by 32x32x16 products with all loads of a step in its second half: 2,048 tokens, four experts
// each, 104 us, 80 (128 rows; 83); 1,712 99, 64 (256; 71); 1,282 98, 56 (192; 58); 512 58, 47 (128; 48). 64 experts of 1,536 on 4,096, 2,500
// tokens: 496, 391 (192; 403); 1,500 348, 308 (128; 312). (All three in one run, experts chosen at random; how unequally busy they are moves these by a tenth.)
#define TALL_BN 256
#define TALL_W_STAGE (TALL_BN * 64)          // elements
#define TALL_WST 3
#define TALL_XST 2
constexpr int tall_lds_of(int TM) { return (TALL_WST * TALL_W_STAGE + TALL_XST * 32 * TM * 64) * 2; }
template <int EPI, int TM>
__global__ void __launch_bounds__(256)
grouped_tile_kernel(const bf16* __restrict__ A, int lda, const bf16* __restrict__ W, int N, int K, void* __restrict__ Cv, int ldc,
                    const int* __restrict__ order, int top, const int* __restrict__ tile_group,
                    const int* __restrict__ tile_row0, const int* __restrict__ tile_rows, float limit, float alpha, float shift,
                    int tiles, int columns) {
    extern __shared__ __attribute__((aligned(1024))) bf16 tall_lds[];       // [TALL_WST][W_STAGE], then [TALL_XST][X_STAGE]
    constexpr int WST = TALL_WST, XST = TALL_XST, X_STAGE = 32 * TM * 64;
    bf16* const xlds = tall_lds + WST * TALL_W_STAGE;
    // (which tile and block of columns: as in the kernel above)
    const int turn = blockIdx.x / XCDS, run = turn / TILE_RUN * XCDS + blockIdx.x % XCDS;
    const int tile = run / columns * TILE_RUN + turn % TILE_RUN, column = run % columns;
    if (tile >= tiles) return;
    const int group = tile_group[tile];
    if (group < 0) return;
    const int row0 = tile_row0[tile], rows = tile_rows[tile];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, g4 = lane >> 4;
    const int wn = wave >> 1, wm = wave & 1;
    const int F = N / 2, out_cols = EPI == 2 ? F : N;
    const int nsteps = K / 64;
    const size_t wstep = (size_t)(N / 16) * 512;
    constexpr int WL = 4, NLX = TM, NLW = 2 * WL, TN = 8;  // a wave's loads of a step
    const bf16* wsrc[WL];
#pragma unroll
    for (int i = 0; i < WL; ++i) {
        const int blk = wave * WL + i;
        int nb = column * (TALL_BN / 16) + blk, last = N / 16 - 1;
        if (EPI == 2) nb = column * (TALL_BN / 32) + blk / 2, last = F / 16 - 1;
        if (nb > last) nb = last;                          // (a block that exists; its sums are not stored)
        if (EPI == 2 && (blk & 1)) nb += F / 16;
        wsrc[i] = W + (size_t)group * N * K + ((size_t)nb * 64 + lane) * 8;
    }
    const bf16* xsrc[NLX];
#pragma unroll
    for (int i = 0; i < NLX; ++i) {
        const int r = (wave * NLX + i) * 8 + (lane >> 3), m = r < rows ? r : rows - 1;
        const int src = top > 0 ? order[row0 + m] / top : row0 + m;
        xsrc[i] = A + (size_t)src * lda + ((lane & 7) ^ ((r >> 1) & 7)) * 8;
    }
    auto load_x = [&](int step, int stage, int i) {
        hb_load_to_lds(xsrc[i] + (size_t)step * 64, xlds + stage * X_STAGE + (wave * NLX + i) * 512);
    };
    auto load_w = [&](int step, int stage, int i) {
        const int ks = i / WL, w = i % WL;
        hb_load_to_lds(wsrc[w] + ((size_t)step * 2 + ks) * wstep,
                       tall_lds + stage * TALL_W_STAGE + ks * (TALL_BN / 16) * 512 + (wave * WL + w) * 512);
    };
    hb_f32x4 acc[TN][TM];
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) acc[a][b] = hb_f32x4{0.f, 0.f, 0.f, 0.f};
    // (the sums stay in accumulation registers: without this the compiler moves them between the products)
    auto hold = [&]() {
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int b = 0; b < TM; ++b) asm volatile("" : "+a"(acc[a][b]));
    };
    constexpr int NM = TN * TM, NR = TN + TM, SLOTS = NM - 8;
    const int w_lane = lane * 8 + wn * TN * 512;
    const int x_lane = (wm * TM * 16 + r16) * 64, x_swizzle = (r16 >> 1) & 7;
    hb_bf16x8 wv[2][TN], xv[2][TM];                        // [set][block]
    auto mfma_one = [&](int set, int j) {
        const int a = j / TM, b = j % TM;
        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[set][a], xv[set][b], acc[a][b], 0, 0, 0);
    };
    auto read_one = [&](int set, int step, int ks, int idx) {      // (all activations and the first weights are needed first)
        if (idx < TM)
            xv[set][idx] = *(const hb_bf16x8*)(xlds + (step % XST) * X_STAGE + x_lane + idx * 16 * 64 + (((4 * ks + g4) ^ x_swizzle) * 8));
        else
            wv[set][idx - TM] = *(const hb_bf16x8*)(tall_lds + (step % WST) * TALL_W_STAGE + ks * (TALL_BN / 16) * 512 + w_lane + (idx - TM) * 512);
    };
    // between the products j and j + 1 of a k-step: nl loads and NR reads, dealt out over the first SLOTS products
    auto between = [&](int j, int nl, auto&& load, auto&& read) {
        const int no = nl + NR;
        const int from = (j < SLOTS ? j : SLOTS) * no / SLOTS, to = (j + 1 < SLOTS ? j + 1 : SLOTS) * no / SLOTS;
#pragma unroll
        for (int o = from; o < to; ++o) {
            const int loads_before = o * nl / no, loads_after = (o + 1) * nl / no;
            if (loads_after > loads_before) load(loads_before);
            else read(o - loads_before);
        }
    };
    auto clamp = [&](int step) { return step < nsteps ? step : nsteps - 1; };   // past the end: the last step again
    // in flight before the loop: steps 0 and 1
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int i = 0; i < NLX; ++i) load_x(clamp(s), s, i);
#pragma unroll
        for (int i = 0; i < NLW; ++i) load_w(clamp(s), s, i);
    }
    hb_wait_vmcnt<NLX + NLW>();
    hb_workgroup_barrier();
#pragma unroll
    for (int i = 0; i < NR; ++i) read_one(0, 0, 0, i);
    hold();
    // (the last step is one like any other: what it loads and reads ahead nobody uses)
    for (int t = 0; t < nsteps; ++t) {
        const int ahead = clamp(t + 2);
        // the first half of a step; its weights of two steps on go into the stage that step t - 1 left at its barrier
#pragma unroll
        for (int j = 0; j < NM; ++j) {
            mfma_one(0, j);
            between(j, NLW, [&](int i) { load_w(ahead, (t + 2) % WST, i); }, [&](int i) { read_one(1, t, 1, i); });
            __builtin_amdgcn_sched_barrier(0);
        }
        // step t + 1 has landed (in flight at most those weights) and, after the barrier, nobody reads step t any more
        hb_wait_vmcnt<NLW>();
        hb_workgroup_barrier();
#pragma unroll
        for (int j = 0; j < NM; ++j) {
            mfma_one(1, j);
            between(j, NLX, [&](int i) { load_x(ahead, t % XST, i); }, [&](int i) { read_one(0, t + 1, 0, i); });
            __builtin_amdgcn_sched_barrier(0);
        }
        hold();
    }
    hb_wait_vmcnt<0>();      // the loads past the end (repeats of the last step) have landed too
    hb_workgroup_barrier();
    // A lane holds runs of four columns of rows 16 b + r16: through LDS of the wave's own, so that whole rows leave. Rows of CH
    // 16-byte chunks, chunk c of row r at c ^ (r mod CH).
    constexpr int COLS = EPI == 2 ? 64 : 128;              // the wave's output columns
    constexpr int PER = EPI == 0 ? 4 : 8;                  // columns a chunk
    constexpr int CH = COLS / PER, RPI = 64 / CH;          // chunks of a row, rows an instruction
    char* const stage = (char*)tall_lds + wave * (32 * CH * 16);       // 32 rows at a time
    static_assert(4 * 32 * CH * 16 <= tall_lds_of(TM), "the waves' rows fit the LDS");
    const int rrow = lane / CH, rchunk = lane % CH;
    const int n = column * (EPI == 2 ? TALL_BN / 2 : TALL_BN) + wn * COLS + rchunk * PER;
#pragma unroll
    for (int b0 = 0; b0 < TM; b0 += 2) {
#pragma unroll
        for (int b = b0; b < b0 + 2; ++b) {
            __builtin_amdgcn_sched_barrier(0);             // (a block of rows after the other: all at once take more registers than there are)
#pragma unroll
            for (int a = 0; a < TN; a += EPI == 2 ? 2 : 1) {
                hb_f32x4 v = acc[a][b];
                if (EPI == 2) {                            // a block of gate rows, then one of their up rows
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const float g = fminf(v[i], limit), u = fminf(fmaxf(acc[a + 1][b][i], -limit), limit);
                        v[i] = g / (1.0f + expf(-alpha * g)) * (u + shift);
                    }
                }
                const int row = 16 * (b - b0) + r16, col = (EPI == 2 ? 8 : 16) * a + 4 * g4;
                char* const at = stage + (row * CH + ((col / PER) ^ (row & (CH - 1)))) * 16;
                if (EPI == 0) {
                    *(hb_f32x4*)at = v;
                } else {
                    bf16 o[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[i] = hb_from_float<bf16>(v[i]);
                    *(uint2*)(at + (col % PER) * 2) = uint2{o[0].bits | ((unsigned)o[1].bits << 16), o[2].bits | ((unsigned)o[3].bits << 16)};
                }
            }
        }
#pragma unroll
        for (int i = 0; i < 32 / RPI; ++i) {
            const int row = i * RPI + rrow, m = (wm * TM + b0) * 16 + row;
            const uint4 v = *(const uint4*)(stage + (row * CH + (rchunk ^ (row & (CH - 1)))) * 16);
            if (m < rows && n < out_cols)                  // (columns come in whole blocks of 16)
                *(uint4*)((char*)Cv + ((size_t)(row0 + m) * ldc + n) * (EPI == 0 ? 4 : 2)) = v;
        }
    }
}

// hb_grouped_mfma for a list of tiles of up to tile_m rows (128, 192 or 256), K in steps of 64, C in rows of whole 16 bytes.
extern "C" int hb_grouped_tall(const void* A, int lda, const void* W, int N, int K, void* C, int ldc, int epi, const int* order,
                               int top, const int* tile_group, const int* tile_row0, const int* tile_rows, int tiles,
                               int tile_m, float limit, float alpha, float shift, hipStream_t stream) {
    HB_REQUIRE(N > 0 && K > 0 && K % 64 == 0, "grouped product: K = %d must be a positive multiple of 64", K);
    HB_REQUIRE(N % 16 == 0 && (epi != 2 || N % 32 == 0), "grouped product: %d weight rows are no whole blocks of 16", N);
    HB_REQUIRE(epi >= 0 && epi <= 2, "grouped product: unknown epilogue %d", epi);
    HB_REQUIRE(lda % 8 == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0 && ldc % (epi == 0 ? 4 : 8) == 0 && (uintptr_t)C % 16 == 0,
               "grouped product: operands must lie at multiples of 16 bytes");
    HB_REQUIRE(tile_m == 128 || tile_m == 192 || tile_m == 256, "grouped product: row tiles of %d", tile_m);
    HB_REQUIRE(tile_group && tiles > 0 && tiles <= 65535, "grouped product: %d row tiles exceed the grid", tiles);
    const int out_cols = epi == 2 ? N / 2 : N, per = epi == 2 ? TALL_BN / 2 : TALL_BN, columns = (out_cols + per - 1) / per;
    const long long runs = (long long)((tiles + TILE_RUN - 1) / TILE_RUN) * columns;
    const long long blocks = (runs + XCDS - 1) / XCDS * XCDS * TILE_RUN;
    HB_REQUIRE(blocks < (1ll << 24), "grouped product: %d tiles of %d columns exceed the grid", tiles, out_cols);
#define HB_TALL(E, TM)                                                                                                      \
    do {                                                                                                                    \
        constexpr int lds = tall_lds_of(TM);                                                                                \
        const hipError_t e_ = hipFuncSetAttribute((const void*)grouped_tile_kernel<E, TM>, hipFuncAttributeMaxDynamicSharedMemorySize, lds); \
        HB_REQUIRE(e_ == hipSuccess, "grouped product: cannot have %d bytes of LDS: %s", lds, hipGetErrorString(e_));        \
        grouped_tile_kernel<E, TM><<<(unsigned)blocks, 256, lds, stream>>>((const bf16*)A, lda, (const bf16*)W, N, K, C, ldc, order, top, \
            tile_group, tile_row0, tile_rows, limit, alpha, shift, tiles, columns);                                          \
    } while (0)
#define HB_TALL_OF(E)                       \
    do {                                    \
        if (tile_m == 128) HB_TALL(E, 4);   \
        else if (tile_m == 192) HB_TALL(E, 6); \
        else HB_TALL(E, 8);                 \
    } while (0)
    if (epi == 0) HB_TALL_OF(0);
    else if (epi == 1) HB_TALL_OF(1);
    else HB_TALL_OF(2);
#undef HB_TALL_OF
#undef HB_TALL
    HB_CHECK_LAUNCH("grouped_tall");
    return 0;
}

// The same for tiles of few rows (decoding), a product bound by the weights' bytes: the four waves of a workgroup take a
// quarter of k each for the same two blocks of weight rows, every operand straight from memory, GS_AHEAD steps of 32 k in
// flight while the GS_AHEAD before are multiplied; the quarters meet in LDS and are added in the waves' order. With all
// of k in a wave a step of four tokens (16 pairs, 13 of 32 experts of 768 on 2,048) took 45 us gate/up and 16 us down,
// each wave a chain of 64 steps with four in flight; now 21 and 14 (75 and 38 MB). 32 tokens: 56 and 25 us, now 38 and 22
// (5.2 TB/s).
#define GS_AHEAD 4
template <int EPI>
__global__ void __launch_bounds__(256)
grouped_mfma_stream_kernel(const bf16* __restrict__ A, int lda, size_t a_group_off, const bf16* __restrict__ W, int N,
                    int K, void* __restrict__ Cv, int ldc, size_t c_group_off, const int* __restrict__ order,
                    int top, const int* __restrict__ tile_group, const int* __restrict__ tile_row0,
                    const int* __restrict__ tile_rows, int M, int m_tiles, float limit, float alpha, float shift) {
    int group, row0, rows;
    if (tile_group) {
        group = tile_group[blockIdx.y];
        if (group < 0) return;
        row0 = tile_row0[blockIdx.y];
        rows = tile_rows[blockIdx.y];
    } else {
        group = blockIdx.y / m_tiles;
        row0 = (blockIdx.y % m_tiles) * MOE_TILE_M;
        rows = M - row0 < MOE_TILE_M ? M - row0 : MOE_TILE_M;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r16 = lane & 15, g4 = lane >> 4;
    const int F = N / 2;
    const int out_cols = EPI == 2 ? F : N;
    // the first of the workgroup's output columns; its weight rows: [n0, n0 + 32), or with EPI 2 [n0, + 16) and [F + n0, + 16)
    const int n0 = EPI == 2 ? blockIdx.x * 16 : blockIdx.x * 32;
    const bf16* Wg = W + (size_t)group * N * K;
    const size_t kstep = (size_t)(N / 16) * 512;
    const bf16* wrow[2];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        int nb = (EPI == 2 ? (a == 0 ? n0 : F + n0) : n0 + 16 * a) / 16;
        if (nb >= N / 16) nb = N / 16 - 1;           // (read a block that exists; its sums are not stored)
        wrow[a] = Wg + (size_t)nb * 512 + lane * 8;
    }
    const int blocks = (rows + 15) / 16;
    const bf16* xrow[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        int m = b * 16 + r16;
        if (m >= rows) m = rows - 1;
        const int src = top > 0 ? order[row0 + m] / top : row0 + m;
        xrow[b] = A + (size_t)src * lda + (size_t)group * a_group_off + g4 * 8;
    }
    hb_f32x4 acc[2][4];
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = hb_f32x4{0.f, 0.f, 0.f, 0.f};

    const int quarter = (K / 32 + 3) / 4;                 // steps a wave takes
    const int first = wave * quarter, last = min(K / 32, first + quarter);
    hb_bf16x8 w_next[GS_AHEAD][2], x_next[GS_AHEAD];
    auto fetch = [&](int s0) {
#pragma unroll
        for (int d = 0; d < GS_AHEAD; ++d) {
            const int step = min(s0 + d, K / 32 - 1);     // (beyond the last: it once more, not multiplied)
#pragma unroll
            for (int a = 0; a < 2; ++a) w_next[d][a] = *(const hb_bf16x8*)(wrow[a] + (size_t)step * kstep);
            x_next[d] = *(const hb_bf16x8*)(xrow[0] + step * 32);
        }
    };
    if (first < last) fetch(first);
    for (int s0 = first; s0 < last; s0 += GS_AHEAD) {
        hb_bf16x8 wv[GS_AHEAD][2], xv[GS_AHEAD];
#pragma unroll
        for (int d = 0; d < GS_AHEAD; ++d) {
            wv[d][0] = w_next[d][0], wv[d][1] = w_next[d][1];
            xv[d] = x_next[d];
        }
        if (s0 + GS_AHEAD < last) fetch(s0 + GS_AHEAD);
#pragma unroll
        for (int d = 0; d < GS_AHEAD; ++d) {
            if (s0 + d >= last) break;
#pragma unroll
            for (int a = 0; a < 2; ++a) acc[a][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[d][a], xv[d], acc[a][0], 0, 0, 0);
#pragma unroll
            for (int b = 1; b < 4; ++b)
                if (b < blocks) {
                    const hb_bf16x8 x = *(const hb_bf16x8*)(xrow[b] + (s0 + d) * 32);
#pragma unroll
                    for (int a = 0; a < 2; ++a) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[d][a], x, acc[a][b], 0, 0, 0);
                }
        }
    }
    __shared__ __attribute__((aligned(16))) hb_f32x4 parts[4][4][2][HB_WAVE];
#pragma unroll
    for (int b = 0; b < 4; ++b)
        if (b < blocks) {
#pragma unroll
            for (int a = 0; a < 2; ++a) parts[wave][b][a][lane] = acc[a][b];
        }
    __syncthreads();
    // wave b adds up and stores the block of rows b
    if (wave >= blocks) return;
#pragma unroll
    for (int a = 0; a < 2; ++a)
        acc[a][0] = ((parts[0][wave][a][lane] + parts[1][wave][a][lane]) + parts[2][wave][a][lane]) + parts[3][wave][a][lane];
    // lane: activation row wave * 16 + r16, weight rows g4 * 4 + i of each block
    const int m = wave * 16 + r16;
    if (m >= rows) return;
    const size_t base = (size_t)(row0 + m) * ldc + (size_t)group * c_group_off;
    if (EPI == 2) {
        bf16* C = (bf16*)Cv;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int n = n0 + g4 * 4 + i;
            if (n >= F) continue;
            const float g = fminf(acc[0][0][i], limit);
            const float u = fminf(fmaxf(acc[1][0][i], -limit), limit);
            C[base + n] = hb_from_float<bf16>(g / (1.0f + expf(-alpha * g)) * (u + shift));
        }
    } else {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int n = n0 + 16 * a + g4 * 4 + i;
                if (n >= N) continue;
                if (EPI == 0)
                    ((float*)Cv)[base + n] = acc[a][0][i];
                else
                    ((bf16*)Cv)[base + n] = hb_from_float<bf16>(acc[a][0][i]);
            }
    }
}

// tile_group null: `groups` groups of ceil(M / 64) tiles each over the same M rows; else a list of
// n_tiles tiles (a group < 0 ends a tile at once). K in steps of 32; lda, a_group_off and the matrices
// such that every operand's 8 numbers lie at a multiple of 16 bytes.
extern "C" int hb_grouped_mfma(const void* A, int lda, size_t a_group_off, const void* W, int N, int K, void* C,
                               int ldc, size_t c_group_off, int epi, const int* order, int top,
                               const int* tile_group, const int* tile_row0, const int* tile_rows, int n_tiles, int M,
                               int groups, float limit, float alpha, float shift, int few_rows, hipStream_t stream) {
    HB_REQUIRE(N > 0 && K > 0 && K % 32 == 0, "grouped product: K = %d must be a positive multiple of 32", K);
    HB_REQUIRE(N % 16 == 0 && (epi != 2 || N % 32 == 0), "grouped product: %d weight rows are no whole blocks of 16", N);
    HB_REQUIRE(lda % 8 == 0 && a_group_off % 8 == 0 && ((uintptr_t)A % 16) == 0 && ((uintptr_t)W % 16) == 0,
               "grouped product: operands must lie at multiples of 16 bytes");
    HB_REQUIRE(epi >= 0 && epi <= 2 && (epi != 2 || N % 2 == 0), "grouped product: unknown epilogue %d", epi);
    int m_tiles = 0, tiles = n_tiles;
    if (!tile_group) {
        HB_REQUIRE(M > 0 && groups > 0 && top == 0, "grouped product: empty batch");
        m_tiles = (M + MOE_TILE_M - 1) / MOE_TILE_M;
        tiles = m_tiles * groups;
    }
    HB_REQUIRE(tiles > 0 && tiles <= 65535, "grouped product: %d row tiles exceed the grid", tiles);
    const int out_cols = epi == 2 ? N / 2 : N;
    // few_rows: the tiles hold few rows each (the host knows how many rows there are to how many groups)
    const int per_group = few_rows ? (epi == 2 ? 16 : 32) : (epi == 2 ? 128 : 256);
    const dim3 grid((out_cols + per_group - 1) / per_group, tiles);
#define HB_GROUPED_STREAM(E)                                                                                        \
    grouped_mfma_stream_kernel<E><<<grid, 256, 0, stream>>>((const bf16*)A, lda, a_group_off, (const bf16*)W, N, K, \
                                                            C, ldc, c_group_off, order, top, tile_group, tile_row0,  \
                                                            tile_rows, M, m_tiles, limit, alpha, shift)
    if (few_rows) {
        if (epi == 0) HB_GROUPED_STREAM(0);
        else if (epi == 1) HB_GROUPED_STREAM(1);
        else HB_GROUPED_STREAM(2);
        HB_CHECK_LAUNCH("grouped_mfma_stream");
        return 0;
    }
#undef HB_GROUPED_STREAM
    const int quads = ldc % 4 == 0 && c_group_off % 4 == 0 && (uintptr_t)C % 16 == 0;
    const long long runs = (long long)((tiles + TILE_RUN - 1) / TILE_RUN) * grid.x;
    const long long blocks = (runs + XCDS - 1) / XCDS * XCDS * TILE_RUN;
    // (a grid's x holds fewer than 2^32 threads: 65,535 tiles of 255 blocks of columns, whose sums no card holds)
    HB_REQUIRE(blocks < (1ll << 24), "grouped product: %d tiles of %d columns exceed the grid", tiles, out_cols);
#define HB_GROUPED(E)                                                                                               \
    grouped_mfma_kernel<E><<<(unsigned)blocks, 256, 0, stream>>>((const bf16*)A, lda, a_group_off, (const bf16*)W, N, K, C, ldc, \
                                                       c_group_off, order, top, tile_group, tile_row0, tile_rows, M, \
                                                       m_tiles, limit, alpha, shift, tiles, (int)grid.x, quads)
    if (epi == 0) HB_GROUPED(0);
    else if (epi == 1) HB_GROUPED(1);
    else HB_GROUPED(2);
#undef HB_GROUPED
    HB_CHECK_LAUNCH("grouped_mfma");
    return 0;
}
