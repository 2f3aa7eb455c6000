"""State-space layers in chunks of 64 tokens (csrc/recurrent_chunks.hip) against the rule token by token in float64 and against
the walk: the edges of chunks and of their blocks of 16, several sequences beside short ones, a state carried over several
launches, decays from one to zero, and rows that are not finite."""
import types

import pytest
import torch

from herbert_rs_amd.kernels import recurrent
from herbert_rs_amd.parts import Runtime

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def step(lengths, heads, groups, N, P, rate, seed=0):
    g = torch.Generator().manual_seed(seed)
    T, B = sum(lengths), len(lengths)
    u = torch.randn(T, heads * P + 2 * groups * N, generator=g)
    proj = torch.randn(T, heads + 5, generator=g)
    a_log, dt_bias, d_skip = (0.5 * torch.randn(heads, generator=g) for _ in range(3))
    starts = torch.tensor([0] + lengths).cumsum(0).to(torch.int32)
    meta = types.SimpleNamespace(max_new=max(lengths), num_seqs=B, seq_starts=starts.to(DEV), host_starts=starts.numpy(), derived={},
                                 slots=torch.arange(B, 0, -1, dtype=torch.int32, device=DEV))
    state = 0.3 * torch.randn(B + 2, heads, P, N, generator=g)        # (as the kernels keep it: a column's entries side by side)
    return u, proj, a_log + rate, dt_bias, d_skip, state, meta


def run(u, proj, a_log, dt_bias, d_skip, state, meta, heads, groups, N, P, chunks=True):
    out, held = torch.full((u.shape[0], heads * P), 7.0, device=DEV), state.to(DEV).reshape(state.shape[0], heads, P * N).contiguous()
    rt = Runtime(torch.float32, DEV) if chunks else None
    recurrent.ssm_scan(u.to(DEV), proj.to(DEV), 5, dt_bias.to(DEV), a_log.to(DEV), d_skip.to(DEV), held, meta, out, heads, groups, N, P, rt=rt)
    assert not chunks or any(name == "ssm_pairs" for name, _ in rt._buffers), "the step did not go through in chunks"
    return out.cpu().view(-1, heads, P), held.cpu().view(state.shape)


def expected(u, proj, a_log, dt_bias, d_skip, state, lengths, heads, groups, N, P):
    outs, states, at = [], state.double().clone(), 0
    for b, n in enumerate(lengths):
        rows, S = u[at:at + n].double(), states[len(lengths) - b]                     # [heads, P, N]
        x = rows[:, :heads * P].view(n, heads, P)
        B, C = (rows[:, heads * P + i * groups * N:][:, :groups * N].view(n, groups, N).repeat_interleave(heads // groups, 1) for i in (0, 1))
        dt = torch.nn.functional.softplus(proj[at:at + n, 5:].double() + dt_bias.double())
        a = torch.exp(-torch.exp(a_log.double()) * dt)
        for t in range(n):
            S = a[t][:, None, None] * S + (dt[t][:, None] * x[t])[:, :, None] * B[t][:, None, :]
            outs.append((S * C[t][:, None, :]).sum(-1) + d_skip.double()[:, None] * x[t])
        states[len(lengths) - b] = S
        at += n
    return torch.stack(outs), states


@pytest.mark.parametrize("rate", [-6.0, -2.0, 0.0, 4.0])       # decays near one, spread over (0, 1), near zero
@pytest.mark.parametrize("lengths,heads,groups,N,P", [([130], 4, 2, 128, 64), ([64, 1, 200, 47, 48, 63, 65], 6, 3, 64, 16),
                                                      ([97, 129, 0], 4, 4, 128, 48), ([1000], 2, 1, 64, 32), ([70] * 9, 3, 1, 128, 16)])
def test_chunks_follow_the_rule(lengths, heads, groups, N, P, rate, monkeypatch):
    """Outputs and the state left, once in one pair of launches and once in several. Sums of up to 128 products and as many
    tokens in float32, a few of them in a row: 2e-6 of a sequence's norm, and no further off than the walk but for a tenth."""
    case = step(lengths, heads, groups, N, P, rate)
    want, want_state = expected(*case[:6], lengths, heads, groups, N, P)
    walk, walk_state = run(*case, heads, groups, N, P, chunks=False)
    for scratch in (recurrent.CHUNK_SCRATCH, 1):               # (1: a chunk a launch)
        monkeypatch.setattr(recurrent, "CHUNK_SCRATCH", scratch)
        got, state = run(*case, heads, groups, N, P)
        for a, b, w in ((got, want, walk), (state, want_state, walk_state)):
            off, walked = float((a - b).norm() / b.norm()), float((w - b).norm() / b.norm())
            print(f"off {off:.2e}, the walk {walked:.2e}")
            assert off <= 2e-6 and off <= 1.1 * walked + 1e-8
        at = 0
        for n in lengths:
            if n:
                assert float((got[at:at + n] - want[at:at + n]).norm() / want[at:at + n].norm()) <= 2e-6, (n, scratch)
            at += n
        assert torch.equal(state[0], case[5][0]) and torch.equal(state[-1], case[5][-1])      # nobody's slots


@pytest.mark.parametrize("place", ["x", "B", "C", "dt", "state"])
@pytest.mark.parametrize("what", [float("nan"), float("inf"), -float("inf"), 3e38])
def test_what_is_not_finite_reaches_what_it_reaches_in_the_walk(place, what):
    """In the middle of a sequence's second chunk (the state: one entry of one head): finite where the walk is finite, and there
    near it; the other sequence is untouched."""
    heads, groups, N, P, lengths = 4, 2, 64, 48, [200, 100]
    u, proj, a_log, dt_bias, d_skip, state, meta = step(lengths, heads, groups, N, P, -1.0)
    t = 64 + 21
    if place == "x":
        u[t, P + 5] = what
    elif place == "B":
        u[t, heads * P + N + 3] = what
    elif place == "C":
        u[t, heads * P + groups * N + 7] = what
    elif place == "dt":
        proj[t, 5 + 2] = what
    else:
        state[2, 1, 3, 9] = what
    case = (u, proj, a_log, dt_bias, d_skip, state, meta)
    got, after = run(*case, heads, groups, N, P)
    walk, walk_after = run(*case, heads, groups, N, P, chunks=False)
    for a, b in ((got, walk), (after, walk_after)):
        assert torch.equal(a.isfinite(), b.isfinite())
        fine = b.isfinite()
        assert float((a - b)[fine].abs().max()) <= 1e-4 * float(b[fine].abs().max())


@pytest.mark.parametrize("place", ["x", "B", "C", "state"])
@pytest.mark.parametrize("rate", [0.0, 1.0])
@pytest.mark.parametrize("what", [1e16, 1e22, 1e30])
def test_large_numbers_pass_no_range_that_they_do_not_pass_in_the_walk(place, what, rate):
    """A state of 1e20 and an input whose product with it, with another input or with a later one passes float32's range before the
    decays bring it back, or only after they have: finite where the walk is, and there near it."""
    heads, groups, N, P, lengths = 4, 2, 64, 48, [200, 100]
    u, proj, a_log, dt_bias, d_skip, state, meta = step(lengths, heads, groups, N, P, rate)
    state[2, 1] *= 1e20
    for t in (50, 64 + 21):
        at = {"x": P + 5, "B": heads * P + 3, "C": heads * P + groups * N + 7, "state": None}[place]
        if at is not None:
            u[t, at] = what
    if place == "state":
        state[2, 1, 3, 9] = what
        u[40, heads * P + groups * N:] *= 1e20               # (C of a token whose decays bring the state far down)
    case = (u, proj, a_log, dt_bias, d_skip, state, meta)
    got, after = run(*case, heads, groups, N, P)
    walk, walk_after = run(*case, heads, groups, N, P, chunks=False)
    for a, b in ((got, walk), (after, walk_after)):
        assert torch.equal(a.isfinite(), b.isfinite())
        fine = b.isfinite()
        assert float((a - b)[fine].abs().max()) <= 1e-4 * float(b[fine].abs().max())


@pytest.mark.parametrize("bad", [False, True])
@pytest.mark.parametrize("lengths,heads,groups,N,P", [([64, 130, 65], 96, 3, 64, 16), ([70, 1000], 65, 5, 128, 48), ([129, 64], 129, 1, 64, 32)])
def test_a_sequence_alone_and_beside_others(lengths, heads, groups, N, P, bad):
    """Few workgroups take 16 columns of the state each and many 32 (the columns' last ones may be half of that): a sequence has the same bits
    either way, also where an entry of B has a chunk walked token by token."""
    u, proj, a_log, dt_bias, d_skip, state, meta = step(lengths, heads, groups, N, P, -2.0)
    if bad:
        u[lengths[0] - 3, heads * P + 7] = float("inf")
    assert heads * ((P + 31) // 32) * len(lengths) > 256 >= heads * ((P + 31) // 32)
    got, left = run(u, proj, a_log, dt_bias, d_skip, state, meta, heads, groups, N, P)
    at = 0
    for b, n in enumerate(lengths):
        slot = len(lengths) - b
        one = types.SimpleNamespace(max_new=n, num_seqs=1, seq_starts=torch.tensor([0, n], dtype=torch.int32, device=DEV), derived={},
                                    host_starts=torch.tensor([0, n], dtype=torch.int32).numpy(), slots=torch.tensor([slot], dtype=torch.int32, device=DEV))
        alone, alone_left = run(u[at:at + n], proj[at:at + n], a_log, dt_bias, d_skip, state, one, heads, groups, N, P)
        assert torch.equal(alone.nan_to_num(7.0), got[at:at + n].nan_to_num(7.0))
        assert torch.equal(alone_left[slot].nan_to_num(7.0), left[slot].nan_to_num(7.0))
        at += n


@pytest.mark.parametrize("place", ["x", "state"])
@pytest.mark.parametrize("what", [float("inf"), 1e20])
@pytest.mark.parametrize("lengths,heads,groups,N,P", [([64, 130, 65], 96, 3, 64, 64), ([70, 1000], 65, 5, 128, 48), ([129, 64], 129, 1, 64, 32)])
def test_a_large_column_alone_and_beside_others(lengths, heads, groups, N, P, what, place):
    """One column's input or state is too large for the products, so that its 16 columns are walked: also in a workgroup of 32, whose other 16 are
    not. The same bits either way, and in those other 16 the bits that they have without the large one."""
    u, proj, a_log, dt_bias, d_skip, state, meta = step(lengths, heads, groups, N, P, -2.0)
    plain, plain_left = run(u, proj, a_log, dt_bias, d_skip, state, meta, heads, groups, N, P)
    if place == "x":
        u[lengths[0] - 3, P + 21] = what
    else:
        state[len(lengths), 1, 21, 9] = what
    assert heads * ((P + 31) // 32) * len(lengths) > 256 >= heads * ((P + 31) // 32)
    got, left = run(u, proj, a_log, dt_bias, d_skip, state, meta, heads, groups, N, P)
    n, slot = lengths[0], len(lengths)
    one = types.SimpleNamespace(max_new=n, num_seqs=1, seq_starts=torch.tensor([0, n], dtype=torch.int32, device=DEV), derived={},
                                host_starts=torch.tensor([0, n], dtype=torch.int32).numpy(), slots=torch.tensor([slot], dtype=torch.int32, device=DEV))
    alone, alone_left = run(u[:n], proj[:n], a_log, dt_bias, d_skip, state, one, heads, groups, N, P)
    assert torch.equal(alone.nan_to_num(7.0), got[:n].nan_to_num(7.0))
    assert torch.equal(alone_left[slot].nan_to_num(7.0), left[slot].nan_to_num(7.0))
    assert not torch.equal(got[:n, 1, 21], plain[:n, 1, 21])
    assert torch.equal(got[:, :, :16], plain[:, :, :16]) and torch.equal(left[:, :, :16], plain_left[:, :, :16])
