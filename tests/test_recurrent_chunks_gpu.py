"""The delta rule and the linear attention in chunks of 64 tokens (csrc/recurrent_chunks.hip) against the rule token by token
in float64: the edges of chunks and of their blocks of 16, several sequences, a head's keys shared, decays from one to zero, a
state that is carried over several launches, and rows that are not finite."""
import types

import pytest
import torch

pytestmark = pytest.mark.gpu


def dev():
    return torch.device("cuda", 0)


def rule(q, k, v, beta, decay, S):
    """q, k, decay [T, H, D], v [T, H, V], beta [T, H] or None, S [H, D, V]: (outputs, last state), token by token."""
    out = []
    for t in range(q.shape[0]):
        S = S * decay[t][:, :, None]
        u = v[t] if beta is None else beta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
        S = S + k[t][:, :, None] * u[:, None, :]
        out.append((S * q[t][:, :, None]).sum(1))
    return torch.stack(out) if out else v, S


def step(lengths, kv_heads, heads, D, V, kind, rate, seed=0):
    """A step of sequences of these lengths; kind "head" or "channel" (the delta rule's decay) or "linear"."""
    g = torch.Generator().manual_seed(seed)
    T, B, W = sum(lengths), len(lengths), 2 * kv_heads * D + heads * V + 4

    def draw(*shape):
        return torch.randn(*shape, generator=g)
    qkv = draw(T, W if kind == "linear" else W - 4)        # (the linear attention reads the columns of a wider row)
    for a in (0, kv_heads * D):
        part = qkv[:, a:a + kv_heads * D].view(T, kv_heads, D)
        part /= part.norm(dim=-1, keepdim=True)
    proj, a_log, dt_bias = draw(T, 2 * heads + 3), 0.5 * draw(heads) + rate, 0.5 * draw(heads)
    decay = torch.exp(-torch.exp(a_log)[:, None] * torch.nn.functional.softplus(draw(T, heads, D)))
    if rate > 2:
        decay[::5] = 0.0                                   # a memory that is dropped at once
    starts = torch.tensor([0] + lengths).cumsum(0).to(torch.int32)
    meta = types.SimpleNamespace(max_new=max(lengths), num_seqs=B, seq_starts=starts.to(dev()), host_starts=starts.numpy(), derived={},
                                 slots=torch.arange(B, 0, -1, dtype=torch.int32, device=dev()))
    state = 0.3 * draw(B + 2, heads, D, V)
    return qkv, proj, a_log, dt_bias, decay, state, meta


def run(qkv, proj, a_log, dt_bias, decay, state, meta, kv_heads, heads, D, V, kind, out_scale=0.5):
    from herbert_rs_amd.kernels import recurrent
    from herbert_rs_amd.parts import Runtime
    rt, T = Runtime(torch.float32, dev()), qkv.shape[0]
    out, held = torch.full((T, heads * V), 7.0, device=dev()), state.to(dev())
    d = None if kind == "head" else decay.reshape(T, heads * D).to(dev())
    recurrent.gated_delta(qkv.to(dev()), None if kind == "linear" else proj.to(dev()), 0, heads, a_log.to(dev()),
                          dt_bias.to(dev()), held, meta, out, kv_heads, heads, D, V, decay=d, correction=kind != "linear",
                          out_scale=out_scale, rt=rt)
    assert any(name == "delta_chunks" for name, _ in rt._buffers), "the step did not go through in chunks"
    return out.cpu().view(T, heads, V), held.cpu()


def expected(qkv, proj, a_log, dt_bias, decay, state, lengths, kv_heads, heads, D, V, kind, out_scale=0.5):
    outs, states, at = [], state.double().clone(), 0
    for b, n in enumerate(lengths):
        rows = qkv[at:at + n].double()
        rep = heads // kv_heads
        q, k = (rows[:, a:a + kv_heads * D].view(n, kv_heads, D).repeat_interleave(rep, 1) for a in (0, kv_heads * D))
        v = rows[:, 2 * kv_heads * D:2 * kv_heads * D + heads * V].view(n, heads, V)
        p = proj[at:at + n].double()
        beta = None if kind == "linear" else torch.sigmoid(p[:, :heads])
        g = decay[at:at + n].double() if kind != "head" else torch.exp(
            -torch.exp(a_log.double()) * torch.nn.functional.softplus(p[:, heads:2 * heads] + dt_bias.double()))[:, :, None].expand(n, heads, D)
        slot = len(lengths) - b
        o, states[slot] = rule(q, k, v, beta, g, states[slot])
        outs.append(o * out_scale)
        at += n
    return torch.cat(outs), states


@pytest.mark.parametrize("kind", ["head", "channel", "linear"])
@pytest.mark.parametrize("rate", [-5.0, 0.0, 4.0])             # decays near one, spread over (0, 1), near zero and zero
@pytest.mark.parametrize("lengths,kv_heads,heads,D,V", [([130], 2, 2, 128, 32), ([64, 1, 200, 16, 63], 2, 6, 64, 16), ([97, 129], 1, 4, 128, 48)])
def test_chunks_follow_the_rule(lengths, kv_heads, heads, D, V, kind, rate, monkeypatch):
    """Outputs and the state left, once in one pair of launches and once in several. float32 sums of up to 128 products of
    numbers of unit size, a few of them in a row: 2e-6 of a sequence's norm (seen: 8e-7)."""
    from herbert_rs_amd.kernels import recurrent
    case = step(lengths, kv_heads, heads, D, V, kind, rate)
    want, want_state = expected(*case[:6], lengths, kv_heads, heads, D, V, kind)
    monkeypatch.setattr(recurrent, "chunks_from", lambda *_: 1)        # (whatever is faster: every portion here)
    for scratch in (recurrent.CHUNK_SCRATCH, 1):               # (1: a chunk a launch)
        monkeypatch.setattr(recurrent, "CHUNK_SCRATCH", scratch)
        got, state = run(*case, kv_heads, heads, D, V, kind)
        at = 0
        for n in lengths:
            assert float((got[at:at + n] - want[at:at + n]).norm() / want[at:at + n].norm()) <= 2e-6, (n, scratch)
            at += n
        assert float((state - want_state).norm() / want_state.norm()) <= 2e-6
        assert torch.equal(state[0], case[5][0]) and torch.equal(state[-1], case[5][-1])      # nobody's slots


@pytest.mark.parametrize("kind", ["head", "channel", "linear"])
@pytest.mark.parametrize("lengths", [[1, 200, 1, 0, 130, 1], [60, 20, 300, 96, 3, 47] + [64] * 30, [64] * 70 + [1]])
def test_long_portions_take_chunks_beside_short_ones(kind, lengths, monkeypatch):
    """Portions that go through in chunks, single tokens and a walk of what lies between in one step, with room for all chunks in
    one call and for a few: the scratch stays within its bound and every sequence follows the rule."""
    from herbert_rs_amd.kernels import recurrent
    from herbert_rs_amd.parts import Runtime
    kv_heads, heads, D, V = 2, 4, 64, 16
    case = step(lengths, kv_heads, heads, D, V, kind, 0.0)
    want, want_state = expected(*case[:6], lengths, kv_heads, heads, D, V, kind)
    room = recurrent.chunk_floats(D, V, kind != "linear") * heads * 7
    for scratch in (recurrent.CHUNK_SCRATCH, room):
        monkeypatch.setattr(recurrent, "CHUNK_SCRATCH", scratch)
        sizes = []
        monkeypatch.setattr(Runtime, "buffer", lambda rt, name, shape, dtype=None, take=Runtime.buffer: sizes.append(shape) or take(rt, name, shape, dtype))
        got, state = run(*case, kv_heads, heads, D, V, kind)
        monkeypatch.undo()
        assert sizes and max(n for n, in sizes) <= scratch
        assert float((got - want).norm() / want.norm()) <= 2e-6 and float((state - want_state).norm() / want_state.norm()) <= 2e-6
        at = 0
        for n in lengths:
            if n:
                assert float((got[at:at + n] - want[at:at + n]).norm() / want[at:at + n].norm()) <= 2e-6, (n, scratch)
            at += n


@pytest.mark.parametrize("kind", ["head", "channel", "linear"])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("decay", [None, 0.5, 0.9, 0.99, 0.999])       # (None: spread over (0, 1))
@pytest.mark.parametrize("cosine", [0.0, 0.8])
def test_chunks_are_as_close_to_the_rule_as_the_walk(kind, D, decay, cosine):
    """Keys drawn at random and keys that resemble each other, decays about a value: the outputs' error against 64 bits is no
    larger than the walk's; the state's no larger by more than a tenth (seen: 1.06 of the walk's, both below 1.1e-7 there)."""
    from herbert_rs_amd.kernels import recurrent
    lengths, heads, V = [233], 8, 48
    qkv, proj, a_log, dt_bias, decays, state, meta = step(lengths, heads, heads, D, V, kind, 0.0, seed=D)
    g = torch.Generator().manual_seed(7)
    if cosine:
        keys = qkv[:, heads * D:2 * heads * D].view(233, heads, D)
        base = torch.randn(heads, D, generator=g).abs()
        keys.copy_((1 - cosine) ** 0.5 * keys + cosine ** 0.5 * base / base.norm(dim=-1, keepdim=True))
        keys /= keys.norm(dim=-1, keepdim=True)
    if decay is not None:
        rate = -2.0 * torch.log(torch.tensor(decay))
        decays = torch.exp(-rate * torch.rand(233, heads, D, generator=g))
        a_log, dt_bias = torch.zeros(heads), torch.zeros(heads)
        proj[:, heads:2 * heads] = torch.log(torch.expm1(rate * torch.rand(233, heads, generator=g).clamp(min=1e-4)))
    case = (qkv, proj, a_log, dt_bias, decays, state)
    want, want_state = expected(*case, lengths, heads, heads, D, V, kind)
    got, left = run(*case, meta, heads, heads, D, V, kind)
    out, held = torch.empty(233, heads * V, device=dev()), state.to(dev())
    recurrent.gated_delta(qkv.to(dev()), None if kind == "linear" else proj.to(dev()), 0, heads, a_log.to(dev()), dt_bias.to(dev()), held,
                          meta, out, heads, heads, D, V, decay=None if kind == "head" else decays.reshape(233, heads * D).to(dev()),
                          correction=kind != "linear", out_scale=0.5)
    assert float((got - want).norm()) <= float((out.cpu().view(233, heads, V) - want).norm())
    assert float((left - want_state).norm()) <= 1.1 * float((held.cpu() - want_state).norm())


@pytest.mark.parametrize("kind", ["head", "channel", "linear"])
@pytest.mark.parametrize("place", [3, 64 + 17])
@pytest.mark.parametrize("what", ["query", "key", "value"])
def test_a_number_that_is_not_finite_reaches_what_it_reaches_in_the_walk(kind, place, what):
    """A query spoils its own token's output, a value its column from there on, a key its head from there on: exactly what the
    walk token by token loses is lost (of the linear attention's state, after a key, all rows for one that no later output
    is without). All else is the same bits as without it."""
    from herbert_rs_amd.kernels import recurrent
    kv_heads, heads, D, V, lengths = 2, 2, 64, 32, [150, 112]
    case = list(step(lengths, kv_heads, heads, D, V, kind, 0.0))
    clean, state = run(*case, kv_heads, heads, D, V, kind)
    case[0] = case[0].clone()
    at = {"query": D + 5, "key": (kv_heads + 1) * D + 5, "value": 2 * kv_heads * D + V + 5}[what]         # of head 1
    case[0][place, at] = float("inf")
    got, left = run(*case, kv_heads, heads, D, V, kind)

    qkv, proj, a_log, dt_bias, decay, held, meta = case
    out, held = torch.full((262, heads * V), 7.0, device=dev()), held.to(dev())
    recurrent.gated_delta(qkv.to(dev()), None if kind == "linear" else proj.to(dev()), 0, heads, a_log.to(dev()), dt_bias.to(dev()), held,
                          meta, out, kv_heads, heads, D, V, decay=None if kind == "head" else decay.reshape(262, heads * D).to(dev()),
                          correction=kind != "linear", out_scale=0.5)
    fine, fine_state = out.cpu().view(262, heads, V).isfinite(), held.cpu().isfinite()
    assert torch.equal(got.isfinite(), fine) and torch.equal(got[fine], clean[fine])
    if kind == "linear" and what == "key":
        assert not fine_state[2, 1].all()
        fine_state[2, 1] = False
    assert torch.equal(left.isfinite(), fine_state) and torch.equal(left[fine_state], state[fine_state])


@pytest.mark.parametrize("kv_heads,heads,D,V", [(1, 1, 1, 4), (2, 4, 33, 36), (3, 3, 64, 100), (2, 4, 128, 128), (1, 2, 200, 8), (1, 1, 256, 64),
                                                (2, 2, 48, 37)])
@pytest.mark.parametrize("kind", ["head", "channel", "linear"])
def test_one_token_a_sequence_is_a_step_of_the_walk(kv_heads, heads, D, V, kind):
    """A step that brings at most one token a sequence (one brings none: its state stays) against float64, beside the walk
    that takes longer portions: float32 sums of at most 256 products, a relative error (2-norm) of a few roundings (2^-24)."""
    from herbert_rs_amd.kernels import recurrent
    lengths = [1, 0, 1, 1]
    qkv, proj, a_log, dt_bias, decay, state, meta = step(lengths, kv_heads, heads, D, V, kind, 0.0, seed=D + V)
    want, want_state = expected(qkv, proj, a_log, dt_bias, decay, state, lengths, kv_heads, heads, D, V, kind)
    for longest in (1, 2):
        meta.max_new = longest
        out, held = torch.full((3, heads * V), 7.0, device=dev()), state.to(dev())
        recurrent.gated_delta(qkv.to(dev()), None if kind == "linear" else proj.to(dev()), 0, heads, a_log.to(dev()), dt_bias.to(dev()),
                              held, meta, out, kv_heads, heads, D, V, decay=None if kind == "head" else decay.reshape(3, heads * D).to(dev()),
                              correction=kind != "linear", out_scale=0.5)
        assert float((out.cpu().view(3, heads, V).double() - want).norm() / want.norm()) <= 2e-6, longest
        assert float((held.cpu().double() - want_state).norm() / want_state.norm()) <= 2e-6, longest
        assert torch.equal(held.cpu()[meta.slots[1].item()], state[meta.slots[1].item()])
