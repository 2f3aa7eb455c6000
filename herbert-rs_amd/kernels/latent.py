"""Host side of the attention over latent rows (csrc/attention_latent.hip): what a token writes
(its cache row [latent | rotated part] and its rotated query parts) and the attention itself."""
import numpy as np
import torch

from ..errors import BackendError
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
TARGET_WAVES = 1024        # a decode step's keys are cut into ranges until about this many waves run


# Steps of several tokens a sequence take the kernel whose workgroups share their keys from contexts beyond this on: two
# chunks of 32 keys leave it nothing to share (8 prompts of 64 tokens: 24 us, a wave a token's heads 23; of 20 tokens 32 and
# 26), at 100 tokens it takes 40 us against 51.
PROMPT_FROM = 64


def mfma_takes(cache, rank, rot):
    """True if the matrix-core kernel takes this latent: bfloat16 rows, the latent and the rotated part in
    steps of 32, up to 512 + 128."""
    return (cache.k.dtype == torch.bfloat16 and rank % 32 == 0 and 0 < rank <= 512 and rot % 32 == 0 and rot <= 128
            and cache.page_size % CHUNK == 0)


# What the built keys and values of a step's sequences may take beyond what the other form of the same step takes.
HEADS_BYTES = 256 << 20
HEADS_TILE = 64


def _tiles(meta):
    return sum(-(-int(n) // HEADS_TILE) for n in meta.host_context)


def heads_pay(meta, kv, H, dim, vdim, rank, rot):
    """True if a step's latent attention builds every head's keys and values (latent_attention_heads) instead of scoring on the
    latents: for the sizes that its kernels take, where the estimate of its time is the smaller, in scratch that stays within its
    bound. The estimates: products of the heads' matrices with latents (keys here, tokens there) at 400 TFLOP/s, the
    attentions' own at 600 and 500, and no less than the longest context's chain of tiles, 1.7 us for 64 keys here and 3.2 us
    for 32 there. Microseconds of a whole layer, latents / built, 16 heads of 128 + 64 and 128 on 512: 65 tokens 79 / 47, 300 tokens
    108 / 56, 16 tokens behind 1,000 144 / 64, behind 8,000 805 / 267; 4 heads of 64 + 32 and 64 on 256: 51 / 32, 65 / 35, 93 / 41
    and 528 / 158."""
    if (meta.max_new == 1 or meta.max_context <= PROMPT_FROM or not mfma_takes(kv, rank, rot) or dim not in (64, 128)
            or vdim != dim or rot not in (0, 32, 64) or kv.page_size % HEADS_TILE):
        return False
    new = np.diff(meta.host_starts).astype(np.int64)
    context = meta.host_context.astype(np.int64)
    pairs, T, tiles = int((new * (context - new) + new * (new + 1) // 2).sum()), int(new.sum()), _tiles(meta)
    matrices = 2 * H * rank * (dim + vdim) / 400e6          # (microseconds a row)
    built = tiles * HEADS_TILE * matrices + max(4 * pairs * H * (dim + rot + vdim) / 600e6, meta.max_context / 64 * 1.7)
    latent = T * matrices + max(4 * pairs * H * (2 * rank + rot) / 500e6, meta.max_context / 32 * 3.2)
    scratch = 2 * tiles * HEADS_TILE * (H * (dim + vdim) + rot) + 4 * T * H * rot
    other = T * H * (4 * (rank + rot) + 2 * (rank + dim))
    return built < latent and scratch <= max(other, HEADS_BYTES)


def latent_attention_heads(q, q_off, turned, meta, kv, w_uk, w_uv, out, gate, gate_off, dim, vdim, rank, rot, scale, buffer,
                           sinks=None):
    """out[t, h, :] = softmax over the slot's rows j <= position of (query . [W_uk,h c_j | r_j] * scale) times W_uv,h c_j, times
    sigmoid(gate[t, gate_off + h]) if a gate is given; bfloat16 [T, H vdim]. q f32 [T, ld]: columns [q_off, + H (dim + rot)) are the
    queries, whose rotated parts are read from turned f32 [T, H rot] instead. w_uk [H, dim, rank], w_uv [H, vdim, rank] as
    moe.pack_grouped gives them. Only where heads_pay says so; scratch from `buffer(name, shape, dtype)`."""
    H = w_uk.shape[0]
    T, ld = q.shape
    _check(q, "q", torch.float32, (T, ld))
    _check(turned, "turned", torch.float32, (T, H * rot))
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
    tiles = _tiles(meta)
    keys = buffer("latent_heads_keys", (H, tiles * HEADS_TILE, dim), torch.bfloat16)
    shared = buffer("latent_heads_turned", (tiles * HEADS_TILE, max(rot, 1)), torch.bfloat16)
    values = buffer("latent_heads_values", (H, tiles * HEADS_TILE, vdim), torch.bfloat16)
    lib.call("attention_latent", "hb_latent_attention_heads", q.data_ptr() + 4 * q_off, ld, turned.data_ptr(), kv.k.data_ptr(),
             w_uk.data_ptr(), w_uv.data_ptr(), keys.data_ptr(), shared.data_ptr(), values.data_ptr(), out.data_ptr(), gate_ptr,
             gate_ld, meta.positions.data_ptr(), meta.seq_starts.data_ptr(), meta.context_lens.data_ptr(), meta.num_seqs,
             meta.slots.data_ptr(), kv.page_table.data_ptr(), kv.page_table.shape[1], kv.page_size, tiles, int(meta.max_new), T,
             H, dim, vdim, rank, rot, float(scale), _ptr(sinks), _stream())


def latent_attention_mfma(q_full, meta, cache, out, gate, gate_off, H, rank, rot, scale, buffer, sinks=None):
    """latent_attention_plain on the matrix cores (see mfma_takes). A prompt's tokens share their keys in LDS; a step of one
    token a sequence cuts its keys into ranges, whose partial results lie in scratch from `buffer(name, shape, dtype)`."""
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
    splits, per = 1, 1 << 30
    if meta.max_new == 1:
        # the grid must not depend on the contexts themselves (a recorded step is replayed at others of its bucket)
        chunks = -(-max(meta.context_bucket, meta.max_context) // CHUNK)
        blocks = T * ((H + 15) // 16)
        splits = max(1, min(TARGET_WAVES // blocks, chunks, 64))
        per = -(-chunks // splits)
    part_acc = part_ml = None
    if splits > 1:
        part_acc = buffer("latent_partial", (T * H * splits, rank), torch.float32)
        part_ml = buffer("latent_partial_ml", (T * H * splits, 2), torch.float32)
    prompt = meta.max_new > 1 and meta.max_context > PROMPT_FROM
    if prompt:
        _check(meta.seq_starts, "seq_starts", torch.int32, (meta.num_seqs + 1,))
    lib.call("attention_latent", "hb_latent_attention_mfma", q_full.data_ptr(), cache.k.data_ptr(), out.data_ptr(),
             _ptr(part_acc), _ptr(part_ml), gate_ptr, gate_ld, meta.positions.data_ptr(), meta.seq_of.data_ptr(),
             meta.slots.data_ptr(), cache.page_table.data_ptr(), cache.page_table.shape[1], cache.page_size, T, H,
             rank, rot, float(scale), splits, per, _ptr(sinks),
             meta.seq_starts.data_ptr() if prompt else None, meta.num_seqs if prompt else 0, int(meta.max_new), _stream())
