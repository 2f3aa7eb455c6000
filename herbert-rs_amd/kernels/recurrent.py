"""Host side of the kernels for mixers with state of fixed size (csrc/recurrent.hip): the short
causal convolution with its activation and unit vectors, the gated delta rule, and the gated norm a
head that follows it. Operand checks, then the launch."""
import numpy as np
import torch

from ..errors import BackendError
from ..hosted import send
from . import lib
from .ops import _check, _stream, dtype_code

MAX_TAPS = 16
MAX_KEY_DIM = 256


def conv_silu(proj, taps, conv_state, meta, out, n_unit, unit_dim, n_scaled, scale, unit_eps, n_plain, plain_dim,
              col0=0, bias=None):
    """out[t, c] = silu(sum_j taps[c, j] * input[t - (K - 1) + j, c]) over the C columns of proj (f32 [T, ld])
    from col0 on; inputs from before the step come from conv_state (f32 [slots, K - 1, C]), which is
    then moved on. The first n_unit sections of unit_dim channels become unit vectors (the first
    n_scaled of them times `scale`), the n_plain sections of plain_dim that follow stay as they are (the last
    of them may be shorter). bias f32 [C]: the sums start there."""
    T, ld = proj.shape
    C, K = taps.shape
    if bias is not None:
        _check(bias, "conv bias", torch.float32, (C,))
    _check(proj, "proj", torch.float32, (T, ld))
    _check(taps, "taps", torch.float32, (C, K))
    _check(conv_state, "conv_state", torch.float32, (None, max(K - 1, 1), C))
    _check(out, "out", torch.float32, (T, C))
    _check(meta.seq_of, "seq_of", torch.int32, (T,))
    _check(meta.seq_starts, "seq_starts", torch.int32, (meta.num_seqs + 1,))
    _check(meta.slots, "slots", torch.int32, (meta.num_seqs,))
    if n_unit * unit_dim + n_plain * plain_dim < C or col0 < 0 or ld < col0 + C or not 1 <= K <= MAX_TAPS:
        raise BackendError(f"conv: sections {n_unit} x {unit_dim} + {n_plain} x {plain_dim} do not fit {C} channels "
                           f"of {K} taps")
    lib.call("recurrent", "hb_conv_silu", proj.data_ptr() + 4 * col0, ld, taps.data_ptr(), conv_state.data_ptr(),
             meta.seq_of.data_ptr(), meta.seq_starts.data_ptr(), meta.slots.data_ptr(), out.data_ptr(), T,
             meta.num_seqs, C, K, n_unit, unit_dim, n_scaled, float(scale), float(unit_eps), n_plain, plain_dim,
             None if bias is None else bias.data_ptr(), int(meta.max_new), _stream())


MAX_SSM_STATE = 256


def ssm_state_floats(N, P):
    """Floats of state that the walk's kernel keeps for a head of N rows and P columns (its own layout: every
    thread's numbers side by side, rows and columns rounded up to what its lanes hold). The kernel's entry point
    refuses a state of another size, so the two cannot drift apart unseen."""
    if not 0 < N <= MAX_SSM_STATE or P <= 0:
        raise BackendError(f"state-space walk: a state of {N} x {P}")
    nr, lpc = (4, 4) if N <= 16 else (4, 8) if N <= 32 else (4, 16) if N <= 64 else (8, 16) if N <= 128 else (16, 16)
    cols = 256 // lpc
    return -(-P // cols) * 256 * nr


def ssm_scan(u, proj, dt_off, dt_bias, a_log, d_skip, state, meta, out, heads, groups, N, P, rt=None):
    """The state-space walk of every sequence of the step: u f32 [T, heads P + 2 groups N] (x, B, C as the
    convolution left them), the step sizes' pre-activations in columns [dt_off, + heads) of proj (f32 [T, ld]);
    dt = softplus(. + dt_bias), S <- exp(-exp(a_log) dt) S + dt B x^T, out = S^T C + d_skip x; state f32
    [slots, heads, ssm_state_floats(N, P)] advanced in place (zeros: an empty state), out f32 [T, heads P]. With a Runtime the
    long portions go through in chunks, for the sizes that those kernels take."""
    T = u.shape[0]
    _check(u, "u", torch.float32, (T, heads * P + 2 * groups * N))
    _check(proj, "proj", torch.float32, (T, None))
    for t, name in ((dt_bias, "dt_bias"), (a_log, "A_log"), (d_skip, "D")):
        _check(t, name, torch.float32, (heads,))
    _check(state, "state", torch.float32, (None, heads, ssm_state_floats(N, P)))
    _check(out, "out", torch.float32, (T, heads * P))
    _check(meta.seq_starts, "seq_starts", torch.int32, (meta.num_seqs + 1,))
    _check(meta.slots, "slots", torch.int32, (meta.num_seqs,))
    if heads % groups or not 0 < N <= MAX_SSM_STATE or dt_off < 0 or dt_off + heads > proj.shape[1]:
        raise BackendError(f"state-space walk: {heads} heads in {groups} groups, a state of {N} rows")
    operands = (u.data_ptr(), u.shape[1], proj.data_ptr(), proj.shape[1], int(dt_off), dt_bias.data_ptr(), a_log.data_ptr(),
                d_skip.data_ptr(), state.data_ptr())
    walks = ((None, meta.num_seqs),)
    if (rt is not None and meta.max_new >= SSM_CHUNKS_FROM and N in (64, 128) and P % 16 == 0 and u.shape[1] % 4 == 0
            and u.data_ptr() % 16 == 0 and state.data_ptr() % 16 == 0):
        calls, floats, walks = _ssm_lists(meta, groups)
        pairs = rt.buffer("ssm_pairs", (floats,), torch.float32)
        for runs, n_runs, chunks, n_chunks in calls:
            lib.call("recurrent_chunks", "hb_chunked_ssm", *operands, chunks.data_ptr(), n_chunks, runs.data_ptr(), n_runs,
                     meta.slots.data_ptr(), out.data_ptr(), pairs.data_ptr(), heads, groups, N, P, state.shape[2], _stream())
    for which, n_seqs in walks:
        lib.call("recurrent", "hb_ssm_scan", *operands, meta.seq_starts.data_ptr(), meta.slots.data_ptr(), out.data_ptr(), n_seqs,
                 heads, groups, N, P, state.shape[2], None if which is None else which.data_ptr(), _stream())


def gated_group_norm(o, proj, z_off, weight, out, parts, eps):
    """out = v / rms(v) * weight with v = o * silu(proj[:, z_off ...]), the root mean square taken over each of
    `parts` equal groups of a row by itself; o f32 [T, width], weight f32 [width], out in any dtype."""
    T, width = o.shape
    _check(o, "o", torch.float32, (T, width))
    _check(proj, "proj", torch.float32, (T, None))
    _check(weight, "weight", torch.float32, (width,))
    _check(out, "out", None, (T, width))
    if parts <= 0 or width % parts or z_off < 0 or z_off + width > proj.shape[1]:
        raise BackendError(f"gated norm in groups: {width} columns in {parts} groups")
    lib.call("recurrent", "hb_gated_group_norm", o.data_ptr(), proj.data_ptr(), proj.shape[1], int(z_off),
             weight.data_ptr(), out.data_ptr(), dtype_code(out), T, width, int(parts), float(eps), _stream())


# Portions of many tokens go through in chunks of CHUNK tokens (csrc/recurrent_chunks.hip), shorter ones token by token.
CHUNK = 64
# Scratch of one call, in floats (or one chunk's, if that is more): a step with more chunks than fit goes through in
# several calls, a sequence's state carried from one to the next. (It also stays below the 256 MB memory-side cache, from
# which the second kernel reads what the first has left.)
CHUNK_SCRATCH = 48 << 20


def chunk_floats(D, V, correction):
    """Floats that a chunk of a head takes of the scratch (the kernel refuses another number)."""
    return (3 if correction else 2) * CHUNK * D + CHUNK * CHUNK + (CHUNK * V if correction else 0) + D + V + 4


def chunks_from(portions, heads, correction, channels):
    """The fewest tokens with which one of a step's portions goes through in chunks (channels: a decay a key channel).
    The walk takes 0.4 us a token of the longest portion (0.6 with a decay a channel) while its waves fit the chip; the chunks 42 us
    (54, without the correction 27) and 4 us a chunk. One sequence of 16 heads of 128: 96 tokens 41 against 46 us, with a
    decay a channel 57 either way, without the correction 48 tokens 27 either way. With many such portions or heads the
    walk's waves wait for each other and the chunks still fill the chip: 8 sequences of 32 tokens 58 us either way, of 64 103 against
    60, with a decay a channel 32 tokens 56 against 70 and 64 tokens 96 against 72, without the correction 12 of 20 tokens 64 against 51
    and 8 of 16 37 against 40."""
    few, many = (48, 20) if not correction else (96, 40) if channels else (112, 32)
    if int((portions >= many).sum()) * heads >= 128:
        return many
    return few if portions.max(initial=0) >= few else int(portions.max(initial=0)) + 1


def walks_of(portions, least, heads):
    """The launches of the portions of fewer than `least` tokens, which go token by token: lists of sequences. Single tokens get
    one of their own (a kernel that streams the state, 47 of them 22 us) where they would hold up the walk of the longer
    ones: one of 20 tokens beside 8 single ones takes 22 us so and 34 together, beside 2 of them 21 and 17."""
    ones = [i for i, n in enumerate(portions) if n == 1 < least]
    longer = [i for i, n in enumerate(portions) if 1 < n < least]
    if longer and ones and len(ones) * heads < 64:
        return [sorted(ones + longer)]
    return [w for w in (ones, longer) if w]


def chunk_calls(starts, least, room):
    """Cut the portions of at least `least` tokens into chunks and these into calls of at most `room` chunks. starts: the
    first packed row of each sequence and the last one's end. A call is (runs [n, 4], chunks [m, 2]) as hb_chunked_delta reads
    them, the longest run first; a sequence's calls follow each other in the order of its tokens. Sequences share a call's
    room evenly, what the short ones leave over goes to the long ones, and where there are more sequences than room
    the longest come first."""
    left = sorted((int(n), int(row), i) for i, (n, row) in enumerate(zip(np.diff(starts), starts)) if n >= least)
    calls = []
    while left:
        free, taken, later = room, [], []
        for k, (n, row, seq) in enumerate(left):                  # the shortest first
            take = min(-(-n // CHUNK), free // (len(left) - k))
            free -= take
            tokens = min(n, take * CHUNK)
            if tokens:
                taken.append((tokens, row, seq))
            if tokens < n:
                later.append((n - tokens, row + tokens, seq))
        runs, chunks = [], []
        for tokens, row, seq in sorted(taken, reverse=True):
            runs.append((seq, len(chunks), row, tokens))
            chunks += [(row + a, min(CHUNK, tokens - a)) for a in range(0, tokens, CHUNK)]
        calls.append((runs, chunks))
        left = sorted(later)
    return calls


def _chunk_lists(meta, heads, correction, channels, size):
    """(calls, floats, walks) of the step, made once for all its layers: for each call in chunks the GPU's (runs, their number,
    chunks, their number), the scratch they need, and for each launch of the other portions the GPU's list of sequences, their
    number and the most tokens that one of them brings."""
    key = ("delta_chunks", heads, correction, channels, size, CHUNK_SCRATCH)
    got = meta.derived.get(key)
    if got is None:
        portions = np.diff(meta.host_starts)
        least = chunks_from(portions, heads, correction, channels)
        packed, calls, walks = [], [], []

        def place(numbers):                                    # (16 bytes aligned)
            at = len(packed)
            packed.extend(numbers + [0] * (-len(numbers) % 4))
            return at
        for runs, chunks in chunk_calls(meta.host_starts, least, max(1, CHUNK_SCRATCH // (size * heads))):
            calls.append((place([x for run in runs for x in run]), len(runs), place([x for chunk in chunks for x in chunk]), len(chunks)))
        for which in walks_of(portions, least, heads):
            walks.append((place(which), len(which), int(portions[which].max())))
        on_gpu = send(np.array(packed, dtype=np.int32), meta.seq_starts.device)
        calls = tuple((on_gpu[a:], n, on_gpu[b:], m) for a, n, b, m in calls)
        walks = tuple((on_gpu[a:], n, longest) for a, n, longest in walks)
        need = max((m for _, _, _, m in calls), default=0) * heads * size
        # (the largest half, quarter, ... of the bound that will do: a buffer that is outgrown is replaced by one twice as large)
        floats = CHUNK_SCRATCH
        while floats // 2 >= need and floats > 1:
            floats //= 2
        got = meta.derived[key] = (calls, max(floats, need), walks)
    return got


# Portions of so many tokens of a state-space layer go through in chunks. Microseconds by the walk / in chunks, 64 heads of 128 x 64: one
# sequence of 32 tokens 17 / 22, 48 23 / 22, 64 30 / 22; four of 32 25 / 29, 48 34 / 30; 16 of 32 81 / 78, 48 116 / 82.
SSM_CHUNKS_FROM = 48


def _ssm_lists(meta, groups):
    """As _chunk_lists, for state-space layers of that many groups: (calls, floats, walks)."""
    key = ("ssm_chunks", groups, CHUNK_SCRATCH, SSM_CHUNKS_FROM)
    got = meta.derived.get(key)
    if got is None:
        size, packed = groups * CHUNK * CHUNK, []

        def place(numbers):                                    # (16 bytes aligned)
            at = len(packed)
            packed.extend(numbers + [0] * (-len(numbers) % 4))
            return at
        calls = [(place([x for run in runs for x in run]), len(runs), place([x for chunk in chunks for x in chunk]), len(chunks))
                 for runs, chunks in chunk_calls(meta.host_starts, SSM_CHUNKS_FROM, max(1, CHUNK_SCRATCH // size))]
        short = [i for i, n in enumerate(np.diff(meta.host_starts)) if n < SSM_CHUNKS_FROM]
        walks = [(place(short), len(short))] if short else []
        on_gpu = send(np.array(packed, dtype=np.int32), meta.seq_starts.device)
        need = max(m for _, _, _, m in calls) * size
        floats = CHUNK_SCRATCH
        while floats // 2 >= need:
            floats //= 2
        got = meta.derived[key] = (tuple((on_gpu[a:], n, on_gpu[b:], m) for a, n, b, m in calls), max(floats, need),
                                   tuple((on_gpu[a:], n) for a, n in walks))
    return got


def _rule(rt, qkv, proj, b_off, a_off, a_log, dt_bias, decay, state, meta, out, kv_heads, heads, D, V, correction, out_scale):
    """The long portions in chunks (with a Runtime, for the sizes that those kernels take), the others token by token."""
    operands = (qkv.data_ptr(), qkv.shape[1], None if proj is None else proj.data_ptr(), 0 if proj is None else proj.shape[1],
                b_off, a_off, None if a_log is None else a_log.data_ptr(), None if dt_bias is None else dt_bias.data_ptr(),
                None if decay is None else decay.data_ptr(), state.data_ptr())
    walks = ((None, meta.num_seqs, int(meta.max_new)),)
    if (rt is not None and meta.max_new > 1 and D in (64, 128) and V % 16 == 0 and qkv.shape[1] % 4 == 0
            and qkv.data_ptr() % 16 == 0 and (decay is None or decay.data_ptr() % 16 == 0)):
        size = chunk_floats(D, V, correction)
        calls, floats, walks = _chunk_lists(meta, heads, correction, decay is not None, size)
        scratch = rt.buffer("delta_chunks", (floats,), torch.float32) if calls else None
        for runs, n_runs, chunks, n_chunks in calls:
            lib.call("recurrent_chunks", "hb_chunked_delta", *operands, chunks.data_ptr(), n_chunks, runs.data_ptr(), n_runs,
                     meta.slots.data_ptr(), out.data_ptr(), scratch.data_ptr(), kv_heads, heads, D, V, 1 if correction else 0,
                     float(out_scale), size, _stream())
    for which, n_seqs, longest in walks:
        lib.call("recurrent", "hb_gated_delta", *operands, meta.seq_starts.data_ptr(), meta.slots.data_ptr(), out.data_ptr(),
                 n_seqs, kv_heads, heads, D, V, 1 if correction else 0, float(out_scale), longest,
                 None if which is None else which.data_ptr(), _stream())


def gated_delta(qkv, proj, b_off, a_off, a_log, dt_bias, state, meta, out, kv_heads, heads, D, V, decay=None,
                correction=True, out_scale=1.0, rt=None):
    """The delta rule over every sequence of the step; qkv f32 [T, at least 2 kv_heads D + heads V] (queries,
    keys, values in a row's first columns), proj f32 [T, ld] with column b_off + h (beta's pre-activation) and a_off + h (the
    decay's), state f32 [slots, heads, D, V] advanced in place, out f32 [T, heads V].
    decay f32 [T, heads D]: a factor a key channel, as `channel_decay` leaves it; a_off, a_log and
    dt_bias are then not read (they may be None). correction False (a decay a key channel must be given):
    the linear attention S <- diag(decay) S + k v^T, o = S^T q; proj is then not read (it may be None).
    out_scale: o is multiplied by it.
    rt: a Runtime whose scratch buffers may be used: portions of many tokens then go through in chunks, which differs
    from the walk token by token by float32 rounding."""
    T, C = qkv.shape
    if not correction:
        if decay is None:
            raise BackendError("linear attention: the walk without a correction takes a decay a key channel")
        _check(decay, "decay", torch.float32, (T, heads * D))
        _check(qkv, "qkv", torch.float32, (T, None))
        _check(state, "state", torch.float32, (None, heads, D, V))
        _check(out, "out", torch.float32, (T, heads * V))
        _check(meta.seq_starts, "seq_starts", torch.int32, (meta.num_seqs + 1,))
        _check(meta.slots, "slots", torch.int32, (meta.num_seqs,))
        if heads % kv_heads or not 0 < D <= MAX_KEY_DIM or C < 2 * kv_heads * D + heads * V:
            raise BackendError(f"linear attention: {heads} heads on {kv_heads} key heads of {D} in rows of {C}")
        _rule(rt, qkv, None, 0, 0, None, None, decay, state, meta, out, kv_heads, heads, D, V, False, out_scale)
        return
    if decay is not None:
        _check(decay, "decay", torch.float32, (T, heads * D))
        a_off = 0
    else:
        _check(a_log, "A_log", torch.float32, (heads,))
        _check(dt_bias, "dt_bias", torch.float32, (heads,))
    _check(qkv, "qkv", torch.float32, (T, 2 * kv_heads * D + heads * V))
    _check(proj, "proj", torch.float32, (T, None))
    ld = proj.shape[1]
    if not (0 <= b_off and b_off + heads <= ld and 0 <= a_off and a_off + heads <= ld):
        raise BackendError("delta rule: the gate columns lie outside the projection's rows")
    _check(state, "state", torch.float32, (None, heads, D, V))
    _check(out, "out", torch.float32, (T, heads * V))
    _check(meta.seq_starts, "seq_starts", torch.int32, (meta.num_seqs + 1,))
    _check(meta.slots, "slots", torch.int32, (meta.num_seqs,))
    if heads % kv_heads or not 0 < D <= MAX_KEY_DIM:
        raise BackendError(f"delta rule: {heads} heads on {kv_heads} key heads of {D}")
    given = decay is not None
    _rule(rt, qkv, proj, b_off, a_off, None if given else a_log, None if given else dt_bias, decay, state, meta, out, kv_heads,
          heads, D, V, True, out_scale)


def gated_head_norm(o, proj, g_off, weight, out, heads, V, eps, gate="silu"):
    """out[t, h, :] = o[t, h, :] / rms * weight * gate(proj[t, g_off + h V ...]), gate "silu" or
    "sigmoid"; out in any dtype."""
    if gate not in ("silu", "sigmoid"):
        raise BackendError(f"gated norm: unknown gate {gate!r}")
    T = o.shape[0]
    _check(o, "o", torch.float32, (T, heads * V))
    _check(proj, "proj", torch.float32, (T, None))
    if g_off < 0 or g_off + heads * V > proj.shape[1]:
        raise BackendError("gated norm: the gate columns lie outside the projection's rows")
    _check(weight, "weight", torch.float32, (V,))
    _check(out, "out", None, (T, heads * V))
    lib.call("recurrent", "hb_gated_head_norm", o.data_ptr(), proj.data_ptr(), proj.shape[1], g_off, weight.data_ptr(),
             out.data_ptr(), dtype_code(out), T, heads, V, float(eps), 1 if gate == "sigmoid" else 0, _stream())


def channel_decay(z, z_off, a_log, dt_bias, out, heads, D):
    """out[t, h, d] = exp(-exp(a_log[h]) * softplus(z[t, z_off + h D + d] + dt_bias[h, d])): the delta rule's
    decay a key channel from its pre-activation. z f32 [T, ld]; out f32 [T, heads D], which may be z
    itself (z_off 0, ld = heads D)."""
    T, ld = z.shape
    _check(z, "z", torch.float32, (T, ld))
    _check(out, "out", torch.float32, (T, heads * D))
    _check(a_log, "A_log", torch.float32, (heads,))
    _check(dt_bias, "dt_bias", torch.float32, (heads * D,))
    if z_off < 0 or z_off + heads * D > ld or (out.data_ptr() == z.data_ptr() and (z_off or ld != heads * D)):
        raise BackendError("channel decay: the pre-activations lie outside their rows")
    lib.call("recurrent", "hb_channel_decay", z.data_ptr() + 4 * z_off, ld, a_log.data_ptr(), dt_bias.data_ptr(),
             out.data_ptr(), T, heads, D, _stream())


def filter_state(proj, conv_state, meta, C, K, bias=None):
    """After a step: conv_state (f32 [slots, K - 1, C]) takes the last K - 1 inputs of each sequence, the first C
    columns of proj's rows (f32 [T, ld]) plus bias (f32 [C]) if given. For mixers that filter in a kernel of
    their own."""
    T, ld = proj.shape
    _check(proj, "proj", torch.float32, (T, ld))
    if K <= 1:
        return
    _check(conv_state, "conv_state", torch.float32, (None, K - 1, C))
    _check(meta.seq_starts, "seq_starts", torch.int32, (meta.num_seqs + 1,))
    _check(meta.slots, "slots", torch.int32, (meta.num_seqs,))
    if bias is not None:
        _check(bias, "bias", torch.float32, (C,))
    if ld < C or K > MAX_TAPS:
        raise BackendError(f"filter state: {C} channels of {K} taps in rows of {ld}")
    lib.call("recurrent", "hb_filter_state", proj.data_ptr(), ld, conv_state.data_ptr(), meta.seq_starts.data_ptr(),
             meta.slots.data_ptr(), meta.num_seqs, C, K, None if bias is None else bias.data_ptr(), _stream())


def lru_inputs(proj, bx, by, taps, filter_bias, conv_state, meta, out):
    """The two branches of a gated linear recurrent unit from the projection's rows [x | y] (f32 [T, ld], W
    channels each): out f32 [T, 2 W] = [filter(x + bx) + filter_bias | gelu_tanh(y + by)]; taps f32 [W, K],
    conv_state f32 [slots, K - 1, W] (the inputs with their bias), moved on afterwards."""
    T, ld = proj.shape
    W, K = taps.shape
    _check(proj, "proj", torch.float32, (T, ld))
    _check(taps, "taps", torch.float32, (W, K))
    for t, name in ((bx, "x bias"), (by, "y bias")):
        _check(t, name, torch.float32, (W,))
    if filter_bias is not None:
        _check(filter_bias, "filter bias", torch.float32, (W,))
    _check(conv_state, "conv_state", torch.float32, (None, max(K - 1, 1), W))
    _check(out, "out", torch.float32, (T, 2 * W))
    _check(meta.seq_of, "seq_of", torch.int32, (T,))
    _check(meta.seq_starts, "seq_starts", torch.int32, (meta.num_seqs + 1,))
    _check(meta.slots, "slots", torch.int32, (meta.num_seqs,))
    if ld < 2 * W or not 1 <= K <= MAX_TAPS:
        raise BackendError(f"recurrent unit: rows of {ld} for 2 x {W} channels, {K} taps")
    lib.call("recurrent", "hb_lru_inputs", proj.data_ptr(), ld, bx.data_ptr(), by.data_ptr(), taps.data_ptr(),
             None if filter_bias is None else filter_bias.data_ptr(), conv_state.data_ptr(), meta.seq_of.data_ptr(),
             meta.seq_starts.data_ptr(), meta.slots.data_ptr(), out.data_ptr(), T, meta.num_seqs, W, K, int(meta.max_new),
             _stream())


def lru_scan(ug, gates, r_bias, i_bias, lam, rate, state, meta, out, block):
    """The recurrence of every sequence of the step, channel by channel: with r = sigmoid(r_pre + r_bias),
    i = sigmoid(i_pre + i_bias), a = exp(-rate r softplus(lam)): S <- a S + sqrt(1 - a^2) i u, out = S g, where
    ug f32 [T, 2 W] = [u | g] and gates f32 [T, 2 W] holds, for every block of `block` channels, that block's
    r_pre then its i_pre; state f32 [slots, W] advanced in place; out [T, W] in any dtype. Where a sequence brings
    128 tokens or more (meta.max_new) a kernel first turns `gates` into decays and inputs where they lie (gates is
    overwritten), and the walk is cut into runs that are walked side by side and joined, which differs from the one
    walk by float32 rounding."""
    T, W2 = ug.shape
    W = W2 // 2
    _check(ug, "ug", torch.float32, (T, 2 * W))
    _check(gates, "gates", torch.float32, (T, 2 * W))
    for t, name in ((r_bias, "r bias"), (i_bias, "i bias"), (lam, "lam")):
        _check(t, name, torch.float32, (W,))
    _check(state, "state", torch.float32, (None, W))
    _check(out, "out", None, (T, W))
    _check(meta.seq_starts, "seq_starts", torch.int32, (meta.num_seqs + 1,))
    _check(meta.slots, "slots", torch.int32, (meta.num_seqs,))
    lib.call("recurrent", "hb_lru_scan", ug.data_ptr(), gates.data_ptr(), r_bias.data_ptr(), i_bias.data_ptr(),
             lam.data_ptr(), float(rate), state.data_ptr(), meta.seq_starts.data_ptr(), meta.slots.data_ptr(),
             out.data_ptr(), dtype_code(out), meta.num_seqs, T, W, int(block), int(meta.max_new), _stream())
