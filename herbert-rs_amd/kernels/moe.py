"""Host side of the routed feed-forward's kernels (csrc/moe.hip): routing and grouping, the products
of an expert's rows with its matrices, the activation, and the weighted sum."""
import functools
import math

import torch

from ..errors import BackendError
from . import lib
from .ops import _check, _ptr, _stream, dtype_code

TILE_M = 64
TALL_TILES = (128, 192, 256)           # of the matrix-core product of many rows an expert
MAX_EXPERTS = 1024


@functools.lru_cache(maxsize=1024)
def max_tiles(pairs, experts, rows=TILE_M, shared=0):
    """The length of the list of row tiles for that many (token, expert) pairs and rows of a shared expert."""
    return -(-pairs // rows) + experts + -(-shared // rows)


class Routing:
    """The buffers that routing fills for a step of T tokens: chosen int32 [T, top], weight f32 [T, top],
    order / row_of int32 [T top], the tiles' lists."""

    def __init__(self, ints, weight, T, E, top, real=None, tall=0, shared=False):
        """real: the first `real` of the E experts have matrices (None: all); the others' output is their input.
        tall: 0, or one of TALL_TILES: a second list, of tiles of that many rows.
        shared: every token takes one more expert, the matrices behind the others'; its rows, a token each, follow the pairs'."""
        self.real = E if real is None else int(real)
        self.tall = int(tall)
        self.shared_rows = T if shared else 0
        A, tiles = T * top, max_tiles(T * top, E, shared=self.shared_rows)
        self.rows = A + self.shared_rows
        self.tall_tiles = max_tiles(A, E, self.tall, self.shared_rows) if self.tall else 0
        need = self.ints_needed(T, E, top, tall, shared)
        if ints.numel() < need or ints.dtype != torch.int32:
            raise BackendError("routing: the int32 buffer is too small")
        self.T, self.E, self.top, self.tiles = T, E, top, tiles
        o = 0
        self.chosen, o = ints[o:o + A], o + A
        self.order, o = ints[o:o + self.rows], o + self.rows
        self.row_of, o = ints[o:o + A], o + A
        self.counts, o = ints[o:o + E], o + E
        self.tile_expert, o = ints[o:o + tiles], o + tiles
        self.tile_row0, o = ints[o:o + tiles], o + tiles
        self.tile_rows, o = ints[o:o + tiles], o + tiles
        self.tall_list = ints[o:o + 3 * self.tall_tiles].view(3, -1) if self.tall else None
        self.weight = weight

    @staticmethod
    @functools.lru_cache(maxsize=1024)
    def ints_needed(T, E, top, tall=0, shared=False):
        rows = T if shared else 0
        return 3 * T * top + rows + E + 3 * max_tiles(T * top, E, shared=rows) + (3 * max_tiles(T * top, E, tall, rows) if tall else 0)


def route(logits, bias, routing, scores=False, groups=1, keep=1, score="sigmoid", worth_top=2, renorm=True):
    """logits f32 [T, E] (+ bias f32 [E]) -> routing (see Routing): the largest logits + bias, weighed by a
    softmax over the chosen. The logits' rows may be wider than E (their first E columns count).
    scores=True: s = sigmoid(logit), the choice runs on s + bias within the `keep` best of `groups` equal
    runs of adjacent experts (a group is worth its top two selection values), and the weights are the chosen
    experts' s over their sum. score="softmax": s is the softmax of the logits over all experts; worth_top 1: a
    group is worth its highest selection value alone; renorm False: the weights are the chosen experts' s as they are.
    Experts from routing.real on have no matrices: their pairs' tiles are marked as holding nothing."""
    r = routing
    if score not in ("sigmoid", "softmax") or worth_top not in (1, 2):
        raise BackendError(f"routing: scores are 'sigmoid' or 'softmax', a group is worth its top 1 or 2, not {score!r}, {worth_top}")
    if not 0 < r.real <= r.E:
        raise BackendError(f"routing: {r.real} of {r.E} experts have matrices")
    _check(logits, "logits", torch.float32, (r.T, None))
    ld = logits.shape[1]
    if ld < r.E:
        raise BackendError(f"routing: logits of {ld} columns for {r.E} experts")
    if scores and (groups <= 0 or r.E % groups or not 0 < keep <= groups
                   or r.top > keep * (r.E // groups)):
        raise BackendError(f"routing: {r.top} experts out of {keep} of {groups} groups of {r.E} experts")
    if bias is not None:
        _check(bias, "bias", torch.float32, (r.E,))
    _check(r.weight, "weight", torch.float32, (r.T, r.top))
    if r.E > MAX_EXPERTS or not 0 < r.top <= r.E:
        raise BackendError(f"routing: {r.top} of {r.E} experts")
    lib.call("moe", "hb_moe_route", logits.data_ptr(), _ptr(bias), r.chosen.data_ptr(), r.weight.data_ptr(),
             r.counts.data_ptr(), r.order.data_ptr(), r.row_of.data_ptr(), r.tile_expert.data_ptr(),
             r.tile_row0.data_ptr(), r.tile_rows.data_ptr(), r.T, r.E, r.top, r.tiles, ld, 1 if scores else 0,
             int(groups), int(keep), r.real, 1 if score == "softmax" else 0, int(worth_top), 1 if renorm else 0,
             _ptr(r.tall_list), r.tall, r.tall_tiles, r.shared_rows, _stream())


def gemm_plain(a, w, c, routing, gather):
    """c[row] = a[src(row)] @ w[expert of row]^T for every pair's row; w [E, N, K]; a [T, K] with
    gather (src = the pair's token) or [pairs, K]; c f32 [pairs, N]."""
    r = routing
    E, N, K = w.shape
    _check(w, "w", None, (r.real, N, K))
    _check(a, "a", None, (r.T if gather else r.T * r.top, K))
    _check(c, "c", torch.float32, (r.T * r.top, N))
    lib.call("moe", "hb_moe_gemm_plain", a.data_ptr(), dtype_code(a), w.data_ptr(), dtype_code(w), c.data_ptr(),
             dtype_code(c), r.order.data_ptr(), r.tile_expert.data_ptr(), r.tile_row0.data_ptr(),
             r.tile_rows.data_ptr(), r.tiles, r.top if gather else 0, N, K, _stream())


def activate(gu, act, limit, alpha, shift=1.0):
    """gu f32 [pairs, 2 F] (gate | up) -> act [pairs, F] = g sigmoid(alpha g) (u + shift) with g = min(gate,
    limit), u = clamp(up, -limit, limit). (limit inf, alpha 1, shift 0: silu(gate) up.)"""
    rows, two_f = gu.shape
    _check(gu, "gate_up", torch.float32, (rows, two_f))
    if two_f % 2:
        raise BackendError("moe activation: the input's width must be even")
    _check(act, "act", None, (rows, two_f // 2))
    lib.call("moe", "hb_moe_activate", gu.data_ptr(), act.data_ptr(), dtype_code(act), rows, two_f // 2, float(limit),
             float(alpha), float(shift), _stream())


def combine(y, routing, x, shared=None, gate=None, identity=None):
    """x[t] += sum_j weight[t, j] * y[row of pair (t, j)]; y f32 [pairs, H], x f32 [T, H].
    shared f32 [T, H] with gate = (f32 [T, ld], column): x[t] += sigmoid(gate[t, column]) * shared[t] as well.
    identity [T, H] (float32 or bfloat16): the experts' input rows, which are the output of a pair whose expert has
    no matrices (routing.real and beyond); needed where there are such experts."""
    r = routing
    H = x.shape[1]
    shared_ptr, gate_ptr, gate_ld = _shared_args(r, H, shared, gate)
    _check(y, "y", torch.float32, (r.T * r.top, H))
    _check(x, "x", torch.float32, (r.T, H))
    if r.real < r.E and identity is None:
        raise BackendError("moe combine: experts without matrices need the experts' input rows")
    if identity is not None:
        _check(identity, "identity", None, (r.T, H))
    lib.call("moe", "hb_moe_combine", y.data_ptr(), r.weight.data_ptr(), r.row_of.data_ptr(), x.data_ptr(), r.T,
             r.top, H, shared_ptr, gate_ptr, gate_ld, _ptr(identity) if r.real < r.E else None,
             0 if identity is None else dtype_code(identity), r.chosen.data_ptr(), r.real, _stream())


def _shared_args(r, H, shared, gate):
    if shared is None:
        return None, None, 0
    rows, column = gate
    _check(shared, "shared", torch.float32, (r.T, H))
    _check(rows, "gate", torch.float32, (r.T, None))
    if not 0 <= column < rows.shape[1]:
        raise BackendError("moe combine: the gate's column lies outside its rows")
    return shared.data_ptr(), rows.data_ptr() + 4 * column, rows.shape[1]


# Up to so many tokens combine_norm runs: a decode step's. (Its kernel in csrc/moe.hip is the faster one as far as it was measured, up to
# 512 tokens; larger steps keep the two kernels, and with them the order of their sums of squares.)
COMBINE_NORM_TOKENS = 64


def combine_norm(y, routing, acc, norm_w, eps, x, rows, alpha_next, shared=None, gate=None):
    """`combine` into acc (which then holds the sums only if alpha_next is 0: nobody reads them) and ops.postnorm of them, in one
    kernel: x = sum / rms(sum) * norm_w, rows (or None) = x in its own type, acc = alpha_next x where that is not 0. For up to
    COMBINE_NORM_TOKENS tokens; False, and nothing done, where the kernel does not take the sizes or rows lie off 16-byte borders."""
    r = routing
    T, H = acc.shape
    if T > COMBINE_NORM_TOKENS or H % 4 or H > 8192 or r.real < r.E:
        return False
    shared_ptr, gate_ptr, gate_ld = _shared_args(r, H, shared, gate)
    _check(y, "y", torch.float32, (T * r.top, H))
    _check(acc, "acc", torch.float32, (r.T, H))
    _check(norm_w, "norm weight", torch.float32, (H,))
    _check(x, "x", torch.float32, (T, H))
    if rows is not None:
        _check(rows, "rows", None, (T, H))
    if (y.data_ptr() | acc.data_ptr() | norm_w.data_ptr() | x.data_ptr() | (shared_ptr or 0) | (_ptr(rows) or 0)) % 16:
        return False
    lib.call("moe", "hb_moe_combine_norm", y.data_ptr(), r.weight.data_ptr(), r.row_of.data_ptr(), acc.data_ptr(), T, r.top, H,
             shared_ptr, gate_ptr, gate_ld, norm_w.data_ptr(), float(eps), x.data_ptr(), _ptr(rows),
             dtype_code(x if rows is None else rows), float(alpha_next), _stream())
    return True


EPI_F32, EPI_BF16, EPI_GLU = 0, 1, 2
# Up to so many rows a group the kernel without a stage in LDS runs (decoding). Microseconds of an expert layer's two products
# by it / by the tiles: 32 experts of 768 on 2,048: 8 rows an expert 62 / 76, 16 rows 75 / 78, 20 rows 80 / 79, 32 rows 94 / 80,
# where the line lies; 64 of 1,536 on 4,096: 8 rows 404 / 415, 12 rows 429 / 418, 16 rows 465 / 421; 16 of 512 on 1,024: 16 rows
# 19 / 32, 64 rows 32 / 37. A head's product of rows that all heads share, 16 of 512 x 128: 16 rows 4.4 / 5.4, 64 rows 5.4 / 8.0.
FEW_ROWS = 16
# From so many rows an expert on the kernel of tall tiles takes gate/up. Microseconds by tiles of 64 / of 128 (weights from memory): 32
# experts of 768 on 2,048: 32 rows an expert 58 / 48, 50 rows 59 / 48, 64 rows 57 / 47, 96 rows 63 / 50; 64 of 1,536 on 4,096: 62 rows
# 363 / 310; where fewer than half the CUs get a tile (16 of 512 on 1,024: 64 rows 24 / 23) nothing is gained.
# Down, whose k is short, takes tall tiles from DOWN_ROWS rows and DOWN_STEPS steps of 64 k on, below DOWN_ALWAYS steps only where down_tall
# expects them to be done sooner.
DOWN_STEPS, DOWN_ALWAYS, DOWN_ROWS = 12, 16, 128
TALL_ROWS = 48


def mfma_takes(K, lda, a_group_off=0, N=16):
    """True if the matrix-core kernel takes products of this inner size, layout and N weight rows
    (bfloat16 operands)."""
    return K % 32 == 0 and lda % 8 == 0 and a_group_off % 8 == 0 and N % 16 == 0


def tiles_expected(height, T, rows, experts, shared):
    """The tiles of `height` rows of a step of T tokens whose experts have `rows` rows on average, spread as a random choice spreads them."""
    tiles, k = 1.0, 1
    while k * height < rows + 4.0 * rows ** 0.5:           # more than k tiles: the chance that an expert has more than k height rows
        tiles += 0.5 * math.erfc((k * height - rows) / (2.0 * rows) ** 0.5)
        k += 1
    return experts * tiles + (-(-T // height) if shared else 0)


@functools.lru_cache(maxsize=1024)
def tall_rows(T, top, routed, experts, hidden, inter, shared=False):
    """The rows of a tall tile (0: none) for a step of T tokens, each on `top` of `routed` outputs of the router, the first `experts` of which have
    bfloat16 matrices in the cores' order. Tall tiles from TALL_ROWS rows an expert on, for sizes that they take; of those the one
    that brings the fewest bytes into a CU: rounds of tiles over the CUs times weight and activation rows of a step; and none where the low
    tiles of 64, two to a CU, are expected to be done sooner (a round of theirs as long as one of 284 rows: 64 experts of 1,536 on 4,096,
    four each and a shared one, 800 tokens: 307 us, 353 by tiles of 128; 64 of 1,408 on 2,048, six each and a shared one, 512 tokens 160 and
    157 to 174). An expert's rows are taken to be spread around their mean as a random choice spreads them, and a round to be full at
    nine tenths, since some experts of a model are busier than that. Over 49 layers (8 to 256 experts, 250 to 4,000 tokens) the height
    that this gives is 3.8 % slower than the best one where experts are chosen at random (1.6 with rounds full to the last tile, 6.2 full at
    eight tenths; at worst 16 experts of 2,048, 1,500 tokens: 35) and at 98 layers of unequally busy ones, deviations of 0.4 to 2.6 of the
    mean, 8.9 % (9.7, 7.1; without the low tiles 10.1): there one height for all experts costs a round that is nearly empty more often than
    not. An estimate that averaged the rounds over both kinds of routing was better by a tenth of a layer's time at some token counts and
    worse by as much at others.
    shared: every token takes one more expert."""
    rows = T * top / routed
    if rows < TALL_ROWS or hidden % 64 or inter % 64:
        return 0
    columns = -(-2 * inter // 256)

    def workgroups(height):
        return tiles_expected(height, T, rows, experts, shared) * columns
    cost = {h: math.ceil(workgroups(h) / 256 + 0.1) * (256 + h) for h in TALL_TILES if workgroups(h) >= 128}
    cost[0] = math.ceil(workgroups(TILE_M) / 512 + 0.1) * 540 if cost else 0
    return min(cost, key=cost.get)


@functools.lru_cache(maxsize=1024)
def down_tall(T, top, routed, experts, hidden, inter, shared, height):
    """True if the down product of a layer whose gate/up takes tall tiles of `height` rows takes them too: from DOWN_ALWAYS steps of 64 k on,
    and from DOWN_STEPS on where its rounds of tiles over the CUs are expected to be done before the low tiles', two to a CU. A round of
    `steps` steps takes height / 122 us a step and 8 beside them, one of low tiles 1.75 and 3. Microseconds by low / tall tiles, 32 experts
    of 768 on 2,048, four each: 2,048 tokens 70 / 63 (128 rows), with a shared expert 71 / 80 (192, the low ones here), 1,712 tokens 51 / 44
    (256); from 16 steps on: 64 of 1,536 on 4,096, 2,500 tokens 267 / 235 (192), 16 of 2,048 on 2,048, two each, 3,000 tokens 98 / 91 (192). There the
    estimate, which adds a round for experts busier than the mean, would be wrong where that round does not come: 64 of 1,408 on 2,048, six
    each, 1,400 tokens 123 / 107 (192), 8 of 3,584 on 4,096, two each, 700 tokens 86 / 81 (256)."""
    steps, rows = inter // 64, T * top / routed
    if not height or steps < DOWN_STEPS or rows < DOWN_ROWS:
        return False
    if steps >= DOWN_ALWAYS:
        return True
    columns = -(-hidden // 256)

    def rounds(tile, at_once):
        return math.ceil(tiles_expected(tile, T, rows, experts, shared) * columns / at_once + 0.1)
    return rounds(height, 256) * (height / 122 * steps + 8) < rounds(TILE_M, 512) * (1.75 * steps + 3)


def fold_pays(T, top, experts, hidden, inter):
    """True if a step of T tokens takes a shared expert of the others' size as one more of them: its two products and the kernel between
    them go, and its rows follow the pairs' in the experts' products. Microseconds of a layer with the shared expert's own products /
    folded: 32 experts of 768 on 2,048, four each: 8 tokens 66 / 56, 128 124 / 111, 512 134 / 110, 2,048 249 / 227; 64 of 1,408, six
    each: 128 tokens 253 / 245, 512 307 / 296. In steps of few rows an expert (the form that streams the matrices) a tile of 64 of the
    shared expert's rows reads its matrices again, which a dense product does not: 128 of 768, one each: 512 tokens 156 / 152, 1,024
    200 / 216, 2,048 273 / 315; 256 of 512, eight each: 512 tokens 319 / 312; 64 of 1,536 on 4,096, four each: 32 tokens 304 / 299,
    64 343 / 349, 128 398 / 408, 256 520 / 526, and beyond those steps 512 505 / 461, 1,024 629 / 565."""
    if T * top > FEW_ROWS * experts:
        return True
    if hidden * inter >= 4 << 20:
        return T <= 32
    return -(-T // TILE_M) * hidden * inter <= 13 << 20


def pack_grouped(w):
    """[G, N, K] -> the same values with every W[g] in the matrix cores' operand order [K / 32, N / 16, 64, 8]
    (lane = 16 * (k / 8 % 4) + n % 16): what grouped_mfma reads."""
    G, N, K = w.shape
    if N % 16 or K % 32:
        raise BackendError("packed matrices need N in steps of 16 and K in steps of 32")
    return w.view(G, N // 16, 16, K // 32, 4, 8).permute(0, 3, 1, 4, 2, 5).contiguous().view(G, N, K)


def grouped_mfma(a, lda, a_group_off, w, c, ldc, c_group_off, epi, routing=None, gather=False, M=0, limit=0.0,
                 alpha=0.0, shift=1.0, tall=False):
    """Group g: C[rows, g * c_group_off + n] = sum_k A[src(row), g * a_group_off + k] * w[g][n, k], bfloat16
    operands, float32 sums; w as pack_grouped gives it. With `routing` the rows are the (token, expert) pairs in their experts' order
    (gather: A's rows are the tokens'); without, every group takes the same M rows. epi: EPI_F32 / EPI_BF16
    store C in that type; EPI_GLU: w[g] is [2 F, K] (gate rows, then up rows) and C bfloat16 [*, F] receives
    the experts' activation with `limit`, `alpha` and `shift` (see activate). tall: by the routing's list of tall tiles."""
    G, N, K = w.shape
    _check(a, "a", torch.bfloat16)
    _check(w, "w", torch.bfloat16, (G, N, K))
    _check(c, "c", torch.bfloat16 if epi != EPI_F32 else torch.float32)
    if not mfma_takes(K, lda, a_group_off, N) or (epi == EPI_GLU and N % 32):
        raise BackendError(f"grouped product: K = {K}, rows {lda} apart and groups {a_group_off} apart are not taken")
    out_cols = N // 2 if epi == EPI_GLU else N
    if routing is not None:
        r = routing
        rows_a, rows_c = (r.T if gather else r.rows), r.rows
        if G != r.real + (1 if r.shared_rows else 0):
            raise BackendError("grouped product: one matrix an expert")
        lists = (r.order.data_ptr(), r.top if gather else 0, r.tile_expert.data_ptr(), r.tile_row0.data_ptr(),
                 r.tile_rows.data_ptr(), r.tiles, 0, 0)
        few = r.T * r.top <= FEW_ROWS * r.real          # (on average; the kernels take any tile either way)
    else:
        rows_a = rows_c = M
        lists = (None, 0, None, None, None, 0, M, G)
        few = M <= FEW_ROWS
    if tall and (routing is None or not routing.tall or K % 64 or a_group_off or c_group_off or ldc % 8):
        raise BackendError(f"grouped product: tall tiles refuse K = {K}, rows {ldc} apart or a routing without a list of them")
    if (rows_a - 1) * lda + (G - 1) * a_group_off + K > a.numel() or \
            (rows_c - 1) * ldc + (G - 1) * c_group_off + out_cols > c.numel():
        raise BackendError("grouped product: an operand does not hold every row that is addressed")
    if tall:
        lib.call("moe", "hb_grouped_tall", a.data_ptr(), lda, w.data_ptr(), N, K, c.data_ptr(), ldc, epi, r.order.data_ptr(),
                 r.top if gather else 0, *(part.data_ptr() for part in r.tall_list), r.tall_tiles, r.tall, float(limit),
                 float(alpha), float(shift), _stream())
        return
    lib.call("moe", "hb_grouped_mfma", a.data_ptr(), lda, a_group_off, w.data_ptr(), N, K, c.data_ptr(), ldc,
             c_group_off, epi, *lists, float(limit), float(alpha), float(shift), 1 if few else 0, _stream())
