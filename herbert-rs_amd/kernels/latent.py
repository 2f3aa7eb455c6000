"""Host side of the attention over latent rows (csrc/attention_latent.hip): what a token writes
(its cache row [latent | rotated part] and its rotated query parts) and the attention itself."""
import functools

import numpy as np
import torch

from ..errors import BackendError
from ..hosted import send
from . import lib
from .ops import _check, _ptr, _stream, dtype_code

MAX_RANK = 1024
MAX_ROT = 128


def _check_pages(meta, cache, T, width):
    _check(meta.positions, "positions", torch.int32, (T,))
    _check(meta.seq_of, "seq_of", torch.int32, (T,))
    _check(meta.slots, "slots", torch.int32, (None,))
    _check(cache.page_table, "page_table", torch.int32, (None, None))
    _check(cache.k, "latent pages", None, (None, 1, cache.page_size, width))


def latent_write(proj, q_off, down_off, norm_w, q_full, inv_freq, meta, cache, H, qd, rank, rot, rot_dims, eps,
                 write_cache=True, q_plain=None, queries=None, q_latent=None, turned=None):
    """proj f32 [T, ld]: columns [down_off, + rank + rot) -> the tokens' cache rows (the latent RMS-normed
    with norm_w, the rest rotated); columns [q_off, + H (qd + rot)) are the queries, whose rotated parts
    go into q_full f32 [T, H (rank + rot)] and, if q_plain (bf16 [T, H qd]) is given, whose unrotated
    parts are copied there.
    queries f32 [T, H (qd + rot)]: the queries lie there and not in proj (q_off is not read). q_latent =
    (first column, norm weight f32 [q_rank], c_q [T, q_rank] in the cache's dtype): nothing is done about
    queries, whose own latent, these columns of proj, RMS-normed, goes to c_q instead (q_full is not written)."""
    T, ld = proj.shape
    _check(proj, "proj", torch.float32, (T, ld))
    base = proj.data_ptr()
    q_at, q_ld = base + 4 * q_off, ld
    latent_at, latent_w, c_q = None, None, None
    if q_latent is not None:
        first, latent_w, c_q = q_latent
        _check(latent_w, "query latent's norm", torch.float32, (None,))
        _check(c_q, "c_q", cache.k.dtype, (T, latent_w.shape[0]))
        if first < 0 or first + latent_w.shape[0] > ld or q_plain is not None or queries is not None:
            raise BackendError("latent write: the query latent's columns lie outside the rows, or come with queries")
        H, q_at, latent_at = 0, None, base + 4 * first
    elif queries is not None:
        _check(queries, "queries", torch.float32, (T, H * (qd + rot)))
        q_at, q_ld = queries.data_ptr(), H * (qd + rot)
    elif q_off < 0 or q_off + H * (qd + rot) > ld:
        raise BackendError("latent write: the queries' columns lie outside the projection's rows")
    if down_off < 0 or down_off + rank + rot > ld:
        raise BackendError("latent write: the columns lie outside the projection's rows")
    _check(norm_w, "norm_w", torch.float32, (rank,))
    q_row, q_place = rank + rot, rank
    if H and turned is not None:
        _check(turned, "turned", torch.float32, (T, H * rot))
        q_full, q_row, q_place = turned, rot, 0
    elif H:
        _check(q_full, "q_full", torch.float32, (T, H * (rank + rot)))
    if rot_dims:
        _check(inv_freq, "inv_freq", torch.float32, (rot_dims // 2,))
    if rot_dims % 2 or not 0 <= rot_dims <= rot:
        raise BackendError(f"latent write: {rot_dims} rotated entries of {rot}")
    _check_pages(meta, cache, T, rank + rot)
    if q_plain is not None:
        _check(q_plain, "q_plain", torch.bfloat16, (T, H * qd))
    lib.call("attention_latent", "hb_latent_write", base + 4 * down_off, ld, norm_w.data_ptr(), q_at, q_ld,
             _ptr(q_full), _ptr(q_plain), _ptr(inv_freq), meta.positions.data_ptr(), meta.seq_of.data_ptr(),
             meta.slots.data_ptr(), cache.page_table.data_ptr(), cache.page_table.shape[1], cache.page_size,
             cache.k.data_ptr(), dtype_code(cache.k), T, H, qd, rank, rot, rot_dims, float(eps),
             1 if write_cache else 0, latent_at, 0 if latent_w is None else latent_w.shape[0], _ptr(latent_w), _ptr(c_q),
             q_row, q_place, _stream())


def latent_attention_plain(q_full, meta, cache, out, gate, gate_off, H, rank, rot, scale, sinks=None):
    """out[t, h, :rank] = softmax over the slot's rows j <= position of (q_full[t, h] . row_j * scale)
    times the rows' first `rank` entries, times sigmoid(gate[t, gate_off + h]) if gate (f32 [T, ld]) is given.
    sinks f32 [H]: the softmax's denominator of head h also holds exp(sinks[h])."""
    if sinks is not None:
        _check(sinks, "sinks", torch.float32, (H,))
    T = q_full.shape[0]
    _check(q_full, "q_full", torch.float32, (T, H * (rank + rot)))
    _check(out, "out", cache.k.dtype, (T, H * rank))
    _check_pages(meta, cache, T, rank + rot)
    if rank > MAX_RANK or rot > MAX_ROT:
        raise BackendError(f"latent attention: a latent of {rank} + {rot}, the kernel takes up to {MAX_RANK} + {MAX_ROT}")
    gate_ptr, gate_ld = None, 0
    if gate is not None:
        _check(gate, "gate", torch.float32, (T, None))
        gate_ld = gate.shape[1]
        if gate_off < 0 or gate_off + H > gate_ld:
            raise BackendError("latent attention: the gate's columns lie outside its rows")
        gate_ptr = gate.data_ptr() + 4 * gate_off
    lib.call("attention_latent", "hb_latent_attention_plain", q_full.data_ptr(), cache.k.data_ptr(), out.data_ptr(),
             dtype_code(cache.k), gate_ptr, gate_ld, meta.positions.data_ptr(), meta.seq_of.data_ptr(),
             meta.slots.data_ptr(), cache.page_table.data_ptr(), cache.page_table.shape[1], cache.page_size, T, H,
             rank, rot, float(scale), _ptr(sinks), _stream())


CHUNK = 32
# A decode step's keys are cut into ranges until about so many workgroups of four waves run, one a CU, and into twice as many where a
# range would have more than RANGE_CHUNKS chunks: every range leaves sums that another kernel reads. With 256 / 512 / 1,024 of them, 16 heads of
# 512 + 64, us: 8 tokens at 2,000 keys (2 chunks a range) 19 / 25 / 25, 16 at 1,000 (2) 17 / 23 / 23, 32 at 1,000 (4) 20.5 / 21.7 / 31, 64 at 2,000 (16)
# 44 / 36 / 47, 48 at 300 (2) 19.6 / 18.2 / 21.9; 32 heads, 32 at 4,000 (32) 78 / 55 / 66. Steps of more than 64 workgroups, by this rule with 256 / with
# 512: 128 tokens at 2,000 72 / 78, 200 at 1,500 88 / 92 (at 150 to 1,500 71 / 65), 300 at 700 66 / 69, 400 at 500 55 / 73; 128 heads, 64 at 1,000 99 / 118.
TARGET_WORKGROUPS = 256
RANGE_CHUNKS = 4


# Steps of several tokens a sequence take the kernel whose workgroups share their keys from contexts beyond this on: two
# chunks of 32 keys leave it nothing to share. Microseconds by it / by four waves a token, 16 heads of 512 + 64: one prompt of 64 tokens 32 / 12, of
# 128 38 / 16, of 300 55 / 34; 8 of 64 34 / 19, of 100 42 / 37, of 300 128 / 127; 8 heads of 256 + 64: one of 128 24 / 10, 8 of 64 20 / 9, of 100 22 / 18,
# of 200 31 / 36, 4 of 400 42 / 54. The line lies below where the times meet because only that kernel keeps a later token's number that is not
# finite out of the tokens before it; prompts whose heads' keys are built come by neither.
PROMPT_FROM = 64


def mfma_takes(cache, rank, rot):
    """True if the matrix-core kernel takes this latent: bfloat16 rows, the latent and the rotated part in
    steps of 32, up to 512 + 128."""
    return (cache.k.dtype == torch.bfloat16 and rank % 32 == 0 and 0 < rank <= 512 and rot % 32 == 0 and rot <= 128
            and cache.page_size % CHUNK == 0)


# What the built keys and values that one call leaves in scratch may take beyond what the other form takes for the same
# sequences. (They lie in buffers of their own names, which a process that uses both forms keeps beside the other's; a buffer that has
# become too small is replaced by one at least twice as large, and kept.)
HEADS_BYTES = 256 << 20
HEADS_TILE = 64
HEADS_MOST = 4          # times the other form's work on the chip
RUNS = 3                # of neighbouring sequences that score on the latents beside others: that many calls of their own


def _heads_take(kv, dim, vdim, rank, rot):
    return (mfma_takes(kv, rank, rot) and dim in (64, 128) and vdim == dim and rot in (0, 32, 64)
            and kv.page_size % HEADS_TILE == 0)


@functools.lru_cache(maxsize=4096)
def _sequence_form(new, context, H, dim, rank, rot, most_bytes):
    """For a sequence that brings `new` tokens and holds `context` with them: whether its attention builds every head's keys and values
    (latent_attention_heads) instead of scoring on the latents, and the bytes that either form takes in scratch for it. The two round
    differently (keys and values to bfloat16 here, mapped queries and summed latents there), so the choice is by what the sequence brings
    and holds alone, and a row's result does not depend on what else the step holds.
    It is built where the estimate of its time alone is the smaller and the work that it puts on the chip no more than HEADS_MOST times
    the other's, so that a step of many sequences with a few tokens each behind long contexts does not pay for every one's contexts.
    The estimates: products of the heads' matrices with latents (keys here, tokens there) at 400 TFLOP/s, the attentions' own at 600 and
    500, and alone no less than the context's chain of tiles, 1.7 us for 64 keys here and 3.2 us for 32 there. Microseconds of a layer's
    kernels on the latents / built, 16 heads of 128 + 64 and 128 on 512: prompts of 2 tokens 25 / 27, of 64 41 / 29, 8 of 8 39 / 32, 32 of
    64 124 / 52; 16 tokens behind 1,000 133 / 56 (4.7 times the work: on the latents), 30 behind 1,000 142 / 55, 20 behind 8,192 826 / 253,
    50 behind 4,096: one 444 / 143, 4 450 / 217, 10 452 / 492, 32 944 / 1,423; 8 heads of 128 + 64 on 256: 2 tokens 18 / 24, 32 of 64 61 / 38,
    50 behind 4,096: one 281 / 125, 32 337 / 633. (Of these the prompts of a few tokens alone are built where the latents are ahead, by 2 to 6 us.)"""
    pairs = new * (context - new) + new * (new + 1) // 2
    matrices = 4 * H * rank * dim / 400e6                   # (microseconds a row)
    here, there = 4 * pairs * H * (2 * dim + rot) / 600e6, 4 * pairs * H * (2 * rank + rot) / 500e6
    build, take = context * matrices, new * matrices
    bytes_here = 2 * _tiles(context) * HEADS_TILE * (2 * H * dim + rot) + 4 * new * H * rot
    bytes_there = new * H * (4 * (rank + rot) + 2 * (rank + dim))
    built = (new > 1 and build + here <= HEADS_MOST * (take + there)
             and build + max(here, context / 64 * 1.7) < take + max(there, context / 32 * 3.2)
             and bytes_here <= max(bytes_there, most_bytes))
    return built, bytes_here, bytes_there


def _tiles(context):
    return -(-context // HEADS_TILE)


class Forms:
    """How a step's sequences go through a layer's latent attention. calls: for each call of latent_attention_heads (which, sequences,
    tiles, longest); rest: of those that score on the latents (which, sequences, first row, rows, longest, longest context, apart) for every
    run of neighbours, or of all of them where there are more than RUNS runs (apart: others' rows lie between theirs). `which` is the list of
    the sequences on the GPU, None where it is all of the step's."""

    def __init__(self, calls=(), rest=()):
        self.calls, self.rest = calls, rest


def forms(meta, kv, H, dim, vdim, rank, rot):
    """The step's Forms, worked out once for all layers of these sizes."""
    if meta.max_new == 1 or not _heads_take(kv, dim, vdim, rank, rot):
        return LATENTS
    key = ("latent_forms", H, dim, rank, rot)
    got = meta.derived.get(key)
    if got is None:
        got = meta.derived[key] = _forms(meta, H, dim, rank, rot)
    return got


def _forms(meta, H, dim, rank, rot):
    starts, context = meta.host_starts.tolist(), meta.host_context.tolist()
    new = [b - a for a, b in zip(starts, starts[1:])]
    groups, runs, rest, held, other = [], [], [], 0, 0
    for i, (n, c) in enumerate(zip(new, context)):
        built, here, there = _sequence_form(n, c, H, dim, rank, rot, HEADS_BYTES)
        if built:
            if not groups or held + here > max(HEADS_BYTES, other + there):
                groups.append([])
                held = other = 0
            groups[-1].append(i)
            held, other = held + here, other + there
        elif n:
            if not rest or any(new[rest[-1] + 1:i]):
                runs.append([])
            runs[-1].append(i)
            rest.append(i)
    if not groups:
        return LATENTS
    apart = len(runs) > RUNS
    if apart:
        runs = [rest]
    whole = len(groups) == 1 and len(groups[0]) == len(new)
    packed, places = [], []
    for one in groups + runs:
        places.append(len(packed))
        packed += one
    on_gpu = None if whole else send(np.array(packed, dtype=np.int32), meta.seq_starts.device)
    at = lambda place: None if on_gpu is None else on_gpu[place:]
    calls = tuple((at(place), len(one), sum(_tiles(context[i]) for i in one), max(new[i] for i in one)) for place, one in zip(places, groups))
    left = tuple((at(place), len(one), starts[one[0]], starts[one[-1] + 1] - starts[one[0]], max(new[i] for i in one),
                  max(context[i] for i in one), apart) for place, one in zip(places[len(groups):], runs))
    return Forms(calls, left)


LATENTS = Forms()       # all of the step scores on the latents


def heads_pay(meta, kv, H, dim, vdim, rank, rot):
    """True if a sequence of the step builds its heads' keys and values (see _sequence_form)."""
    return (meta.max_new > 1 and _heads_take(kv, dim, vdim, rank, rot)
            and any(_sequence_form(int(n), int(c), H, dim, rank, rot, HEADS_BYTES)[0]
                    for n, c in zip(np.diff(meta.host_starts), meta.host_context)))


def latent_attention_heads(q, q_off, turned, meta, kv, w_uk, w_uv, out, gate, gate_off, dim, vdim, rank, rot, scale, buffer,
                           sinks=None, call=None, turned_at=None):
    """out[t, h, :] = softmax over the slot's rows j <= position of (query . [W_uk,h c_j | r_j] * scale) times W_uv,h c_j, times
    sigmoid(gate[t, gate_off + h]) if a gate is given; bfloat16 [T, H vdim]. q f32 [T, ld]: columns [q_off, + H (dim + rot)) are the
    queries, whose rotated parts are read from turned f32 [T, H rot] instead, or with turned_at = (floats a head, the first one) from
    there in turned f32 [T, H x floats]. w_uk [H, dim, rank], w_uv [H, vdim, rank] as moe.pack_grouped gives them. call: one of Forms'
    calls (None: all sequences); other sequences' rows of out stay as they are. Scratch from `buffer(name, shape, dtype)`."""
    H = w_uk.shape[0]
    T, ld = q.shape
    _check(q, "q", torch.float32, (T, ld))
    turned_row, turned_first = (rot, 0) if turned_at is None else turned_at
    if turned_first < 0 or turned_first + rot > turned_row:
        raise BackendError("latent attention: the rotated parts lie outside their rows")
    _check(turned, "turned", torch.float32, (T, H * turned_row))
    _check(w_uk, "w_uk", torch.bfloat16, (H, dim, rank))
    _check(w_uv, "w_uv", torch.bfloat16, (H, vdim, rank))
    _check(out, "out", torch.bfloat16, (T, H * vdim))
    _check_pages(meta, kv, T, rank + rot)
    _check(kv.k, "latent pages", torch.bfloat16)
    _check(meta.seq_starts, "seq_starts", torch.int32, (meta.num_seqs + 1,))
    _check(meta.context_lens, "context_lens", torch.int32, (meta.num_seqs,))
    if sinks is not None:
        _check(sinks, "sinks", torch.float32, (H,))
    if q_off < 0 or q_off + H * (dim + rot) > ld:
        raise BackendError("latent attention: the queries' columns lie outside their rows")
    gate_ptr, gate_ld = None, 0
    if gate is not None:
        _check(gate, "gate", torch.float32, (T, None))
        gate_ld = gate.shape[1]
        if gate_off < 0 or gate_off + H > gate_ld:
            raise BackendError("latent attention: the gate's columns lie outside its rows")
        gate_ptr = gate.data_ptr() + 4 * gate_off
    if call is None:
        call = None, meta.num_seqs, sum(_tiles(int(n)) for n in meta.host_context), int(meta.max_new)
    which, n_seqs, tiles, longest = call
    if which is not None and (which.dtype != torch.int32 or which.numel() < n_seqs):
        raise BackendError("latent attention: the list of sequences is too short")
    keys = buffer("latent_heads_keys", (H, tiles * HEADS_TILE, dim), torch.bfloat16)
    shared = buffer("latent_heads_turned", (tiles * HEADS_TILE, max(rot, 1)), torch.bfloat16)
    values = buffer("latent_heads_values", (H, tiles * HEADS_TILE, vdim), torch.bfloat16)
    lib.call("attention_latent", "hb_latent_attention_heads", q.data_ptr() + 4 * q_off, ld, turned.data_ptr() + 4 * turned_first,
             turned_row, kv.k.data_ptr(), w_uk.data_ptr(), w_uv.data_ptr(), keys.data_ptr(), shared.data_ptr(), values.data_ptr(), out.data_ptr(), gate_ptr,
             gate_ld, meta.positions.data_ptr(), meta.seq_starts.data_ptr(), meta.context_lens.data_ptr(), n_seqs,
             meta.slots.data_ptr(), kv.page_table.data_ptr(), kv.page_table.shape[1], kv.page_size, tiles, longest, T,
             H, dim, vdim, rank, rot, float(scale), _ptr(sinks), _ptr(which), _stream())


def latent_attention_mfma(q_full, meta, cache, out, gate, gate_off, H, rank, rot, scale, buffer, sinks=None, part=None):
    """latent_attention_plain on the matrix cores (see mfma_takes). A prompt's tokens share their keys in LDS; a step of one
    token a sequence cuts its keys into ranges, whose partial results lie in scratch from `buffer(name, shape, dtype)`.
    part: one of Forms' `rest`, for those sequences alone (of the rows between its first and last any may be written)."""
    if sinks is not None:
        _check(sinks, "sinks", torch.float32, (H,))
    T = q_full.shape[0]
    _check(q_full, "q_full", torch.float32, (T, H * (rank + rot)))
    _check(out, "out", torch.bfloat16, (T, H * rank))
    _check_pages(meta, cache, T, rank + rot)
    if not mfma_takes(cache, rank, rot):
        raise BackendError(f"latent attention: the matrix-core kernel does not take a latent of {rank} + {rot}")
    gate_ptr, gate_ld = None, 0
    if gate is not None:
        _check(gate, "gate", torch.float32, (T, None))
        gate_ld = gate.shape[1]
        if gate_off < 0 or gate_off + H > gate_ld:
            raise BackendError("latent attention: the gate's columns lie outside its rows")
        gate_ptr = gate.data_ptr() + 4 * gate_off
    which, n_seqs, first, rows, longest, context, apart = part or (None, meta.num_seqs, 0, T, int(meta.max_new), meta.max_context, False)
    prompt = apart or (longest > 1 and context > PROMPT_FROM)
    splits, per = 1, 1 << 30
    if longest == 1 and not prompt:
        # the grid must not depend on the contexts themselves (a recorded step is replayed at others of its bucket)
        chunks = -(-max(meta.context_bucket if part is None else 0, context) // CHUNK)
        blocks = rows * ((H + 15) // 16)
        splits = max(1, min(TARGET_WORKGROUPS // blocks, chunks, 64))
        if -(-chunks // splits) > RANGE_CHUNKS:
            splits = max(1, min(2 * TARGET_WORKGROUPS // blocks, chunks, 64))
        per = -(-chunks // splits)
    part_acc = part_ml = None
    if splits > 1:
        part_acc = buffer("latent_partial", (rows * H * splits, rank), torch.float32)
        part_ml = buffer("latent_partial_ml", (rows * H * splits, 2), torch.float32)
    if prompt:
        # (rows as the sequences' starts count them)
        _check(meta.seq_starts, "seq_starts", torch.int32, (meta.num_seqs + 1,))
        first, rows = 0, T
    if which is not None and (which.dtype != torch.int32 or which.numel() < n_seqs):
        raise BackendError("latent attention: the list of sequences is too short")
    lib.call("attention_latent", "hb_latent_attention_mfma", q_full.data_ptr() + 4 * first * H * (rank + rot), cache.k.data_ptr(),
             out.data_ptr() + 2 * first * H * rank, _ptr(part_acc), _ptr(part_ml),
             None if gate_ptr is None else gate_ptr + 4 * first * gate_ld, gate_ld, meta.positions.data_ptr() + 4 * first,
             meta.seq_of.data_ptr() + 4 * first, meta.slots.data_ptr(), cache.page_table.data_ptr(), cache.page_table.shape[1],
             cache.page_size, rows, H, rank, rot, float(scale), splits, per, _ptr(sinks),
             meta.seq_starts.data_ptr() if prompt else None, n_seqs if prompt else 0, longest, _ptr(which) if prompt else None, _stream())
