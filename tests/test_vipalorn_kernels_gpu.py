"""Each mechanism of the Vipalorn decoder alone on the GPU against its plain formula: the layer norm (also
with a sum added on the way), the short convolution with its state, the delta rule in one piece, in
portions and token by token over slots that are used again, the gated norm a head, the latent rows'
write and the attention over them (plain and matrix cores; a far key that holds the weight, keys at
the edges of pages), routing, the experts' products and their weighted sum."""
import math

import numpy as np
import pytest
import torch

from herbert_rs_amd.cache import Cache, KVNeed, StateNeed
from herbert_rs_amd.engine import batch as batching
from herbert_rs_amd.engine.batch import StepEntry
from herbert_rs_amd.kernels import latent, moe, ops, recurrent

from .plain import vipalorn as plain

pytestmark = pytest.mark.gpu
DEV = "cuda"


def rand(*shape, seed=0, scale=1.0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale


def step_meta(cache, slots, counts):
    entries = [StepEntry(s, [0] * n, []) for s, n in zip(slots, counts)]
    starts = [cache.length(s) for s in slots]
    cache.reserve_all([(s, n) for s, n in zip(slots, counts)])
    meta = batching.pack(entries, starts, torch.device(DEV))
    for s, n in zip(slots, counts):
        cache.commit(s, n)
    return meta


@pytest.mark.parametrize("H", [24, 100, 1536])
def test_layer_norm_and_the_sum_it_adds(H):
    x, w, d = rand(7, H, seed=1), 1 + 0.1 * rand(H, seed=2), rand(7, H, seed=3)
    for dtype, tol in ((torch.float32, 2e-6), (torch.bfloat16, 1.6e-2)):
        xg, y = x.to(DEV).clone(), torch.empty(7, H, dtype=dtype, device=DEV)
        ops.layernorm(xg, w.to(DEV), y, 1e-5)
        assert torch.allclose(y.float().cpu(), plain.layer_norm(x, w, 1e-5), atol=tol * 4, rtol=tol)
        ops.layernorm(xg, w.to(DEV), y, 1e-5, delta=d.to(DEV), mult=0.3)
        assert torch.allclose(xg.cpu(), x + 0.3 * d, atol=1e-6)
        assert torch.allclose(y.float().cpu(), plain.layer_norm(x + 0.3 * d, w, 1e-5), atol=tol * 4, rtol=tol)
    rows = torch.tensor([5, 0, 5], dtype=torch.int32, device=DEV)
    y = torch.empty(3, H, device=DEV)
    ops.layernorm(x.to(DEV), w.to(DEV), y, 1e-5, rows)
    assert torch.allclose(y.cpu(), plain.layer_norm(x[[5, 0, 5]], w, 1e-5), atol=1e-5)
    xg = x.to(DEV).clone()
    ops.layernorm(xg, w.to(DEV), xg, 1e-5)                      # in place
    assert torch.allclose(xg.cpu(), plain.layer_norm(x, w, 1e-5), atol=1e-5)


def delta_reference(proj, taps, a_log, dt_bias, kv_heads, heads, D, V, b_off, a_off):
    """q, k, v after convolution, silu and unit vectors, and the recurrence's outputs, by the plain formulas."""
    T, C = proj.shape[0], 2 * kv_heads * D + heads * V
    y = plain.silu(plain.short_conv(proj[:, :C], taps))
    q = plain.unit_vectors(y[:, :kv_heads * D].view(T, kv_heads, D)) * D ** -0.5
    k = plain.unit_vectors(y[:, kv_heads * D:2 * kv_heads * D].view(T, kv_heads, D))
    v = y[:, 2 * kv_heads * D:].view(T, heads, V)
    beta = plain.sigmoid(proj[:, b_off:b_off + heads])
    decay = torch.exp(-torch.exp(a_log) * plain.softplus(proj[:, a_off:a_off + heads] + dt_bias))
    group = heads // kv_heads
    out = torch.stack([plain.delta_rule(q[:, n // group], k[:, n // group], v[:, n], beta[:, n], decay[:, n])
                       for n in range(heads)], 1)
    return torch.cat([q.reshape(T, -1), k.reshape(T, -1), v.reshape(T, -1)], 1), out.reshape(T, heads * V)


@pytest.mark.parametrize("kv_heads,heads,D,V,K", [(1, 1, 8, 5, 1), (2, 6, 24, 70, 3), (3, 3, 48, 33, 4), (1, 2, 128, 64, 2),
                                                  (1, 1, 200, 12, 5)])
def test_convolution_and_delta_rule_whole_in_portions_and_token_by_token(kv_heads, heads, D, V, K):
    C = 2 * kv_heads * D + heads * V
    ld = C + heads * V + 2 * heads + 3
    b_off, a_off = C + heads * V + 1, C + heads * V + 1 + heads
    lengths = [41, 3, 18]
    taps = (1.0 / K + 0.3 * rand(C, K, seed=5))
    a_log, dt_bias = torch.tensor([-3.0, 0.2, -1.0, 0.5, -5.0, 0.0])[:heads], 0.3 * rand(heads, seed=7)
    projs = [rand(n, ld, seed=10 + i, scale=1.5) for i, n in enumerate(lengths)]
    refs = [delta_reference(p, taps, a_log, dt_bias, kv_heads, heads, D, V, b_off, a_off) for p in projs]
    needs = {0: (StateNeed((heads, D, V)), StateNeed((max(K - 1, 1), C)))}
    cache = Cache(needs, 64 * 8, 4096, torch.float32, DEV, max_slots=4)
    state, conv_state = cache.state_views(0)
    for cuts in ([], [1, 2, 3, 9, 17, 40], list(range(1, 41))):
        slots = [cache.alloc_slot() for _ in lengths]           # (slots that the round before has used: cleared)
        got_qkv = [[] for _ in lengths]
        got_out = [[] for _ in lengths]
        edges = sorted(set([0] + cuts + [max(lengths)]))
        for a, b in zip(edges[:-1], edges[1:]):
            live = [i for i, n in enumerate(lengths) if a < n]
            counts = [min(b, lengths[i]) - a for i in live]
            meta = step_meta(cache, [slots[i] for i in live], counts)
            proj = torch.cat([projs[i][a:a + c] for i, c in zip(live, counts)]).to(DEV).contiguous()
            T = proj.shape[0]
            qkv = torch.empty(T, C, device=DEV)
            recurrent.conv_silu(proj, taps.to(DEV), conv_state, meta, qkv, 2 * kv_heads, D, kv_heads, D ** -0.5, 1e-6, heads, V)
            out = torch.empty(T, heads * V, device=DEV)
            recurrent.gated_delta(qkv, proj, b_off, a_off, a_log.to(DEV), dt_bias.to(DEV), state, meta, out, kv_heads, heads, D, V)
            at = 0
            for i, c in zip(live, counts):
                got_qkv[i].append(qkv[at:at + c].cpu())
                got_out[i].append(out[at:at + c].cpu())
                at += c
        for i in range(len(lengths)):
            assert torch.allclose(torch.cat(got_qkv[i]), refs[i][0], atol=2e-6), f"convolution, cuts {cuts[:4]}"
            assert torch.allclose(torch.cat(got_out[i]), refs[i][1], atol=3e-6), f"delta rule, cuts {cuts[:4]}"
        for s in slots:
            cache.free_slot(s)


@pytest.mark.parametrize("D,units,C,biased", [(64, 3, 3 * 64 + 100, False), (128, 18, 18 * 128 + 4, True), (4, 5, 28, False),
                                              (256, 4, 1024, False), (1, 0, 1540, True)])
def test_convolution_of_quads_is_the_general_ones(D, units, C, biased):
    """Rows of whole quads against rows of odd length (which take a wave a section): the sums and their activation are
    the same operations, so plain sections are the same bits; unit ones differ by the order of their D squares, at most
    (D + 3) roundings of half an ulp each in the sum and half of that in its root. Prompts and single tokens alike."""
    section = min(256, C)
    plain_n = -(-(C - units * D) // section) if C > units * D else 0
    taps, bias = 0.25 + 0.3 * rand(C, 4, seed=5).to(DEV), 0.2 * rand(C, seed=6).to(DEV) if biased else None
    got = []
    for odd in (0, 3):
        cache = Cache({0: (StateNeed((3, C)),)}, 64 * 16, 4096, torch.float32, DEV, max_slots=4)
        conv_state, = cache.state_views(0)
        slots = [cache.alloc_slot() for _ in range(3)]
        outs = []
        for step, counts in enumerate(([1, 1, 1], [300, 2, 11], [1, 1, 1], [1, 1, 1], [7, 1, 3], [1, 1, 1])):
            meta = step_meta(cache, slots, counts)
            T = sum(counts)
            proj = torch.empty(T, C + 8 + odd, device=DEV)
            proj[:, 4:4 + C] = rand(T, C, seed=20 + step, scale=1.5).to(DEV)
            out = torch.empty(T, C, device=DEV)
            recurrent.conv_silu(proj, taps, conv_state, meta, out, units, D, 1, 0.5, 1e-6, plain_n, section, col0=4, bias=bias)
            outs += [out, conv_state[torch.tensor(slots, device=DEV)].clone()]
        got.append(outs)
    for a, b in zip(*got):
        cut = units * D if a.dim() == 2 else 0
        assert torch.equal(a[..., cut:], b[..., cut:])
        assert torch.allclose(a[..., :cut], b[..., :cut], rtol=(D + 6) * 2.0 ** -24, atol=0)


def test_gated_norm_a_head():
    T, heads, V = 5, 3, 70
    o, proj, w = rand(T, heads * V, seed=1), rand(T, heads * V + 9, seed=2), 1 + 0.1 * rand(V, seed=3)
    want = (plain.rms_scale(o.view(T, heads, V), 1e-5) * w * plain.silu(proj[:, 4:4 + heads * V].view(T, heads, V))).reshape(T, -1)
    for dtype, tol in ((torch.float32, 1e-5), (torch.bfloat16, 2e-2)):
        y = torch.empty(T, heads * V, dtype=dtype, device=DEV)
        recurrent.gated_head_norm(o.to(DEV), proj.to(DEV), 4, w.to(DEV), y, heads, V, 1e-5)
        assert torch.allclose(y.float().cpu(), want, atol=tol, rtol=tol)


def latent_reference(proj, positions, norm_w, uk, uv, H, qd, rank, rot, rot_dims, base, scale, eps, gate_off):
    T = proj.shape[0]
    q = proj[:, :H * (qd + rot)].view(T, H, qd + rot)
    down = proj[:, H * (qd + rot):H * (qd + rot) + rank + rot]
    c = plain.rms_scale(down[:, :rank], eps) * norm_w
    r = plain.rotate_half_layout(down[:, rank:], positions, base, rot_dims) if rot else down[:, rank:]
    qr = plain.rotate_half_layout(q[..., qd:], positions, base, rot_dims) if rot else q[..., qd:]
    gate = plain.sigmoid(proj[:, gate_off:gate_off + H])
    pos = torch.as_tensor(positions)
    outs = []
    for n in range(H):
        s = (q[:, n, :qd] @ uk[n].T @ c.T + qr[:, n] @ r.T) * scale        # uk [H, rank, qd]
        s = s.masked_fill(pos[None, :] > pos[:, None], -math.inf)
        outs.append(torch.softmax(s, -1) @ c * gate[:, n:n + 1])
    return torch.cat([c, r], 1), torch.stack(outs, 1).reshape(T, H * rank)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("H,qd,rank,rot,rot_dims", [(3, 8, 24, 8, 4), (16, 32, 96, 32, 32), (20, 16, 128, 64, 64), (2, 8, 40, 0, 0)])
def test_latent_rows_and_attention_with_a_far_key(dtype, H, qd, rank, rot, rot_dims):
    """A prompt of 200 tokens, then tokens one by one to 330 (past the pages' edges at 64, 128, ...), beside a
    short sequence in the same steps. The query of every token is made to point at the latent of one far
    key (position 5, or the key at the last page's first place), so that this key holds most of the weight."""
    base, scale, eps = 5000.0, 0.25, 1e-5
    row, qw = rank + rot, H * (qd + rot)
    ld = qw + row + H
    L = 330
    proj = rand(L, ld, seed=3)
    uk, uv = rand(H, rank, qd, seed=4, scale=0.3), None
    norm_w = 1 + 0.1 * rand(rank, seed=5)
    if dtype == torch.bfloat16:
        proj, uk, norm_w = proj.bfloat16().float(), uk.bfloat16().float(), norm_w
    positions = list(range(L))
    rows_ref, out_ref = latent_reference(proj, positions, norm_w, uk, uv, H, qd, rank, rot, rot_dims, base, scale, eps, qw + row)
    short = 70
    rows_short, out_short = latent_reference(proj[:short] * 0.5, positions[:short], norm_w, uk, uv, H, qd, rank, rot, rot_dims,
                                             base, scale, eps, qw + row)
    store = dtype
    cache = Cache({0: KVNeed(1, row, None, values=False)}, 64 * 8, 4096, store, DEV, max_slots=3)
    kv = cache.kv_view(0)
    inv_freq = (base ** (-2.0 * torch.arange(rot_dims // 2, dtype=torch.float32) / max(rot_dims, 1))).to(DEV) if rot_dims else None
    use_cores = latent.mfma_takes(kv, rank, rot)
    buffers = {}

    def buffer(name, shape, dt):
        return buffers.setdefault((name, tuple(shape)), torch.empty(tuple(shape), dtype=dt, device=DEV))
    a, b = cache.alloc_slot(), cache.alloc_slot()
    got, got_short = [], []
    steps = [(200, short)] + [(1, 0)] * (L - 200)
    done = 0
    for n_long, n_short in steps:
        slots, counts = ([a, b], [n_long, n_short]) if n_short else ([a], [n_long])
        meta = step_meta(cache, slots, counts)
        p = torch.cat([proj[done:done + n_long]] + ([proj[:short] * 0.5] if n_short else [])).to(DEV).contiguous()
        T = p.shape[0]
        q_full = torch.zeros(T, H * row, device=DEV)
        latent.latent_write(p, 0, qw, norm_w.to(DEV), q_full, inv_freq, meta, kv, H, qd, rank, rot, rot_dims, eps)
        ops.gemm_plain_batched(p, uk.to(DEV), q_full, T, rank, qd, ld, qd, H * row, H, qd + rot, rank * qd, row)
        out = torch.empty(T, H * rank, dtype=store, device=DEV)
        if use_cores:
            latent.latent_attention_mfma(q_full, meta, kv, out, p, qw + row, H, rank, rot, scale, buffer)
        else:
            latent.latent_attention_plain(q_full, meta, kv, out, p, qw + row, H, rank, rot, scale)
        got.append(out[:n_long].float().cpu())
        if n_short:
            got_short.append(out[n_long:].float().cpu())
        done += n_long
    tol = 2e-5 if dtype == torch.float32 else 3e-2
    assert torch.allclose(torch.cat(got), out_ref, atol=tol, rtol=tol)
    assert torch.allclose(torch.cat(got_short), out_short, atol=tol, rtol=tol)
    # the cached rows themselves
    table = kv.page_table[a].cpu().tolist()
    stored = torch.cat([kv.k[table[p // 64], 0, p % 64].float().cpu()[None] for p in range(L)])
    assert torch.allclose(stored, rows_ref, atol=1e-5 if dtype == torch.float32 else 2e-2, rtol=1e-2)


def test_a_single_far_key_holds_the_weight():
    """One key among hundreds has a score far above the others: the output is that key's latent (times the gate),
    whichever page it lies in, in the prompt and for single tokens; with one position less the key is unseen."""
    H, rank, rot = 16, 64, 32
    row = rank + rot
    for dtype in (torch.float32, torch.bfloat16):
        cache = Cache({0: KVNeed(1, row, None, values=False)}, 64 * 8, 4096, dtype, DEV, max_slots=2)
        kv = cache.kv_view(0)
        slot = cache.alloc_slot()
        L = 300
        meta = step_meta(cache, [slot], [L])
        rows = rand(L, row, seed=1, scale=0.1).to(dtype)
        table = kv.page_table[slot].cpu().tolist()
        for far in (0, 63, 64, 191, 299):
            rows_far = rows.clone()
            rows_far[far, :rank] = 1.0
            for p in range(L):
                kv.k[table[p // 64], 0, p % 64] = rows_far[p].to(DEV)
            q_full = torch.zeros(L, H * row, device=DEV)
            q_full.view(L, H, row)[:, :, :rank] = 2.0                      # score 2 * 64 * 0.25 = 32 against the far key
            out = torch.empty(L, H * rank, dtype=dtype, device=DEV)
            if latent.mfma_takes(kv, rank, rot):
                latent.latent_attention_mfma(q_full, meta, kv, out, None, 0, H, rank, rot, 0.25, None)
            else:
                latent.latent_attention_plain(q_full, meta, kv, out, None, 0, H, rank, rot, 0.25)
            out = out.float().cpu().view(L, H, rank)
            assert torch.allclose(out[far:], torch.ones(L - far, H, rank), atol=2e-2), f"far key {far} in {dtype}"
            if far:
                assert float(out[far - 1].abs().max()) < 0.5              # just before it: unseen


@pytest.mark.parametrize("H,rank,rot", [(16, 512, 64), (5, 512, 128), (3, 480, 0), (20, 256, 96), (8, 32, 0), (64, 128, 32)])
def test_prompt_tokens_share_their_keys(H, rank, rot):
    """The prompt kernel of the latent attention, whose workgroups take 64 (token, head) rows of a sequence: heads that no tile
    divides, latents of one step to sixteen (odd ones among them), sequences that go on in the
    cache, a sink and a gate, against float64; rows behind the sequences' ends may hold anything. bfloat16 keys as
    stored, queries and weights in 16 bits, an output of 8: 2^-8 of the largest entry."""
    row, held, new = rank + rot, [150, 70, 1, 97], [150, 30, 1, 97]
    cache = Cache({0: KVNeed(1, row, None, values=False)}, 64 * 16, 4096, torch.bfloat16, DEV, max_slots=len(held))
    kv = cache.kv_view(0)
    slots = [cache.alloc_slot() for _ in held]
    for s, n, k in zip(slots, held, new):
        if n > k:
            step_meta(cache, [s], [n - k])
    meta = step_meta(cache, slots, new)
    kv.k.fill_(float("nan"))
    rows = [rand(n, row, seed=i).to(torch.bfloat16) for i, n in enumerate(held)]
    for s, r in zip(slots, rows):
        table = kv.page_table[s].cpu().tolist()
        for p in range(r.shape[0]):
            kv.k[table[p // 64], 0, p % 64] = r[p].to(DEV)
    T = sum(new)
    q, gate, sinks = rand(T, H * row, seed=9), rand(T, H, seed=10), rand(H, seed=11)
    out = torch.empty(T, H * rank, dtype=torch.bfloat16, device=DEV)
    latent.latent_attention_mfma(q.to(DEV), meta, kv, out, gate.to(DEV), 0, H, rank, rot, row ** -0.5, None, sinks=sinks.to(DEV))
    at = 0
    for r, n, k in zip(rows, held, new):
        for t in range(k):
            keys = r[:n - k + t + 1].double()
            score = q[at + t].view(H, row).double() @ keys.T * row ** -0.5
            w = torch.softmax(torch.cat([score, sinks.double()[:, None]], 1), -1)[:, :-1]
            want = (w @ keys[:, :rank]) * torch.sigmoid(gate[at + t].double())[:, None]
            err = (out[at + t].cpu().double().view(H, rank) - want).abs().max()
            assert float(err) <= 2.0 ** -8 * float(want.abs().max()) + 1e-3, (n, t)
        at += k
    # a later token's key without finite numbers, and one that is only larger: the tokens before it are the same bits; those
    # that see it lose at least the numbers that are not finite
    late, table = 140, kv.page_table[slots[0]].cpu().tolist()
    for what in (float("inf"), float("nan"), 40.0):
        kv.k[table[late // 64], 0, late % 64, 7:9] = what
        again = torch.empty_like(out)
        latent.latent_attention_mfma(q.to(DEV), meta, kv, again, gate.to(DEV), 0, H, rank, rot, row ** -0.5, None, sinks=sinks.to(DEV))
        assert torch.equal(again[:late], out[:late]) and torch.equal(again[150:], out[150:])
        if what != 40.0:
            assert not again[late:150].view(10, H, rank)[:, :, 7:9].isfinite().any()


@pytest.mark.parametrize("ranges", [1, 14, 21, 1024])
@pytest.mark.parametrize("H,rank,rot", [(16, 512, 64), (5, 512, 128), (3, 480, 0), (17, 160, 96), (8, 32, 0), (20, 288, 32), (16, 128, 128)])
def test_a_token_a_sequence_by_waves_that_share_a_row(H, rank, rot, ranges, monkeypatch):
    """The latent attention of one token a sequence, whose four waves take a quarter of a row's numbers each: latents and rotated parts
    that no four waves share evenly, one chunk of keys and several at their edges, one range, two to six of several chunks (the later ones empty or
    shorter; twice as many as workgroups were asked for, because their chunks would be too many) and as many as there are chunks,
    a sink and a gate, against float64; the tolerance of the prompts' kernel."""
    row, held = rank + rot, [1, 31, 32, 33, 64, 150, 330]
    given = []
    monkeypatch.setattr(latent, "TARGET_WORKGROUPS", ranges)
    cache = Cache({0: KVNeed(1, row, None, values=False)}, 64 * 24, 4096, torch.bfloat16, DEV, max_slots=len(held))
    kv = cache.kv_view(0)
    slots = [cache.alloc_slot() for _ in held]
    for s, n in zip(slots, held):
        if n > 1:
            step_meta(cache, [s], [n - 1])
    meta = step_meta(cache, slots, [1] * len(held))
    kv.k.zero_()
    rows = [rand(n, row, seed=i).to(torch.bfloat16) for i, n in enumerate(held)]
    for s, r in zip(slots, rows):
        table = kv.page_table[s].cpu().tolist()
        for p in range(0, r.shape[0], 64):
            kv.k[table[p // 64], 0, :min(64, r.shape[0] - p)] = r[p:p + 64].to(DEV)
    q, gate, sinks = rand(len(held), H * row, seed=9), rand(len(held), H, seed=10), rand(H, seed=11)
    out = torch.empty(len(held), H * rank, dtype=torch.bfloat16, device=DEV)

    def buffer(name, shape, dt):
        given.append(shape[0] // (len(held) * H))
        return torch.empty(shape, dtype=dt, device=DEV)
    latent.latent_attention_mfma(q.to(DEV), meta, kv, out, gate.to(DEV), 0, H, rank, rot, row ** -0.5, buffer, sinks=sinks.to(DEV))
    assert set(given) == ({1: set(), 14: {4}, 21: {6}, 1024: {16}} if H <= 16 else {1: set(), 14: {2}, 21: {3}, 1024: {16}})[ranges]
    for t, r in enumerate(rows):
        keys = r.double()
        score = q[t].view(H, row).double() @ keys.T * row ** -0.5
        w = torch.softmax(torch.cat([score, sinks.double()[:, None]], 1), -1)[:, :-1]
        want = (w @ keys[:, :rank]) * torch.sigmoid(gate[t].double())[:, None]
        err = (out[t].cpu().double().view(H, rank) - want).abs().max()
        assert float(err) <= 2.0 ** -8 * float(want.abs().max()) + 1e-3, held[t]


@pytest.mark.parametrize("M", [1, 16, 17, 64, 65, 200, 700])
@pytest.mark.parametrize("G,N,K,pad", [(1, 16, 32, 0), (5, 48, 160, 0), (3, 272, 64, 4), (4, 512, 96, 3)])
def test_grouped_products_of_any_rows(M, G, N, K, pad):
    """A product a group on the matrix cores, every epilogue: rows that fill no tile, more column blocks and tiles than a turn
    over the XCDs and fewer, k that no workgroup's four waves divide, and output rows that start at no whole quad.
    float32 sums of bfloat16 products: K / 2^24 of the terms' sizes."""
    from herbert_rs_amd.kernels import moe
    w, a = rand(G, N, K, seed=1).to(torch.bfloat16), rand(M, G * K, seed=2).to(torch.bfloat16)
    for epi in (moe.EPI_F32, moe.EPI_BF16) + ((moe.EPI_GLU,) if N % 32 == 0 else ()):
        cols = N // 2 if epi == moe.EPI_GLU else N
        off = cols + pad
        c = torch.full((M, G * off), 3.0, dtype=torch.float32 if epi == moe.EPI_F32 else torch.bfloat16, device=DEV)
        moe.grouped_mfma(a.to(DEV), G * K, K, moe.pack_grouped(w.to(DEV)), c, G * off, off, epi, M=M, limit=2.0, alpha=1.702, shift=1.0)
        got = c.cpu().double().view(M, G, off)
        for g in range(G):
            rows = a[:, g * K:(g + 1) * K].double()
            want, size = rows @ w[g].double().T, rows.abs() @ w[g].double().abs().T
            slack = K * 2.0 ** -24 * size + 1e-6
            if epi == moe.EPI_GLU:
                z, u = want[:, :cols].clamp(max=2.0), want[:, cols:].clamp(-2.0, 2.0)
                want, slack = z * torch.sigmoid(1.702 * z) * (u + 1.0), 1e-4
            if epi != moe.EPI_F32:
                slack = slack + want.abs() * 2.0 ** -8
            assert bool(((got[:, g, :cols] - want).abs() <= slack).all()), (epi, g)
            assert bool((got[:, g, cols:] == 3.0).all())


@pytest.mark.parametrize("E,top,groups,keep,score,logit_form", [
    (1, 1, 1, 1, "sigmoid", False), (64, 8, 8, 4, "sigmoid", False), (64, 16, 1, 1, "softmax", True), (65, 3, 5, 2, "softmax", False),
    (128, 8, 1, 1, "sigmoid", False), (130, 65, 1, 1, "sigmoid", True), (200, 5, 200, 7, "sigmoid", False),
    (256, 16, 16, 2, "softmax", False), (300, 6, 3, 1, "sigmoid", False), (1024, 9, 1, 1, "sigmoid", True)])
def test_routing_of_few_tokens_is_the_many_tokens_one(E, top, groups, keep, score, logit_form):
    """The choice is exact: equals by index, zeros of both signs are equals. Steps of 1, 8 and 9 tokens are rows of the
    large step's, bit for bit, and rows, counts and tiles follow from the choice alone."""
    T = 417
    logits = rand(T, E + 1, seed=1, scale=1.5)
    logits[::3] = (logits[::3] * 2).round() / 2             # many equals
    logits[1::7] *= -0.0 if E < 65 else 1.0
    bias = (0.25 * rand(E, seed=2)).round() if E % 2 else None

    def go(rows):
        n = rows.shape[0]
        r = moe.Routing(torch.full((moe.Routing.ints_needed(n, E, top),), -7, dtype=torch.int32, device=DEV),
                        torch.empty(n, top, device=DEV), n, E, top, real=max(1, E - 2))
        moe.route(rows.to(DEV), None if bias is None else bias.to(DEV), r, scores=not logit_form, groups=groups, keep=keep, score=score)
        chosen, pairs = r.chosen.view(n, top).cpu(), n * top
        flat = chosen.flatten().long()
        order = torch.sort(flat, stable=True).indices.int()
        assert torch.equal(r.order.cpu(), order)
        assert torch.equal(r.row_of.cpu()[order.long()], torch.arange(pairs, dtype=torch.int32))
        counts = torch.bincount(flat, minlength=E)
        assert torch.equal(r.counts.cpu().long(), counts)
        tiles, row = [], 0
        for e, c in enumerate(counts.tolist()):
            tiles += [(e if e < r.real else -1, row + i, min(64, c - i)) for i in range(0, c, 64)]
            row += c
        got = list(zip(r.tile_expert.tolist(), r.tile_row0.tolist(), r.tile_rows.tolist()))
        assert got[:len(tiles)] == tiles and all(t[0] == -1 for t in got[len(tiles):])
        return chosen, r.weight.cpu()

    chosen, weight = go(logits)
    if logit_form:
        values = logits[:, :E] + (0 if bias is None else bias)
        assert torch.equal(chosen.long(), torch.sort(-values, dim=-1, stable=True).indices[:, :top])
        assert torch.allclose(weight, torch.softmax(torch.gather(values, 1, chosen.long()), -1), rtol=1e-5, atol=1e-7)
    for a, n in ((0, 1), (1, 8), (9, 9), (18, 3)):
        c, w = go(logits[a:a + n])
        assert torch.equal(c, chosen[a:a + n]) and torch.equal(w, weight[a:a + n])


@pytest.mark.parametrize("T,E,top", [(1, 3, 3), (9, 5, 2), (300, 16, 4), (70, 130, 7)])
def test_routing_groups_and_products(T, E, top):
    W, F = 64, 96                                          # (K in steps of 32: what the matrix-core product takes)
    y, wr, br = rand(T, W, seed=1), rand(E, W, seed=2, scale=0.3), 0.1 * rand(E, seed=3)
    logits = (y @ wr.T).to(DEV).contiguous()
    routing = moe.Routing(torch.empty(moe.Routing.ints_needed(T, E, top), dtype=torch.int32, device=DEV),
                          torch.empty(T, top, device=DEV), T, E, top)
    moe.route(logits, br.to(DEV), routing)
    chosen, weight = plain.route(y, wr, br, top)
    got_chosen = routing.chosen.view(T, top).cpu()
    assert torch.equal(got_chosen.sort(-1).values, chosen.sort(-1).values.int())
    assert torch.allclose(routing.weight.cpu().sort(-1).values, weight.sort(-1).values, atol=1e-6)
    # every pair once, an expert's rows together, the tiles cover them
    order, row_of = routing.order.cpu(), routing.row_of.cpu()
    assert sorted(order.tolist()) == list(range(T * top)) and torch.equal(order[row_of.long()], torch.arange(T * top, dtype=torch.int32))
    experts_in_order = got_chosen.flatten()[order.long()]
    assert torch.equal(experts_in_order, experts_in_order.sort().values)
    gate_up, down = rand(E, 2 * F, W, seed=4, scale=0.2), rand(E, W, F, seed=5, scale=0.2)
    want = torch.zeros(T, W)
    for t in range(T):
        for j in range(top):
            e = int(got_chosen[t, j])
            want[t] += routing.weight[t, j].cpu() * plain.expert(y[t:t + 1], gate_up[e, :F], gate_up[e, F:], down[e], 1.5)[0]
    for dtype, tol in ((torch.float32, 2e-5), (torch.bfloat16, 4e-2)):
        yg, gu_w, down_w = y.to(DEV).to(dtype), gate_up.to(DEV).to(dtype), down.to(DEV).to(dtype)
        act = torch.empty(T * top, F, dtype=dtype, device=DEV)
        out = torch.empty(T * top, W, device=DEV)
        x = torch.zeros(T, W, device=DEV)
        if dtype == torch.bfloat16:
            moe.grouped_mfma(yg, W, 0, moe.pack_grouped(gu_w), act, F, 0, moe.EPI_GLU, routing, gather=True, limit=1.5, alpha=1.702)
            moe.grouped_mfma(act, F, 0, moe.pack_grouped(down_w), out, W, 0, moe.EPI_F32, routing)
        else:
            gu = torch.empty(T * top, 2 * F, device=DEV)
            moe.gemm_plain(yg, gu_w, gu, routing, gather=True)
            moe.activate(gu, act, 1.5, 1.702)
            moe.gemm_plain(act, down_w, out, routing, gather=False)
        moe.combine(out, routing, x)
        assert torch.allclose(x.cpu(), want, atol=tol, rtol=tol), f"{dtype}"
