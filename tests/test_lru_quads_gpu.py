"""The recurrent unit's inputs and decays of prompts, four channels a thread (csrc/recurrent.hip): the same bits as a channel a
thread, which the same rows at an address that is no multiple of 16 bytes still take."""
import types

import pytest
import torch

from herbert_rs_amd.kernels import recurrent

pytestmark = pytest.mark.gpu
DEV = "cuda"


def placed(t, odd):
    """A copy of t that starts 4 bytes past a multiple of 16, or at one."""
    room = torch.empty(t.numel() + 4, device=DEV)
    view = room[1 if odd else 0:][:t.numel()].view(t.shape)
    return view.copy_(t)


@pytest.mark.parametrize("lengths", [[257], [300, 1, 2, 3, 70], [8] * 33 + [128]])
@pytest.mark.parametrize("W,blocks", [(8, 2), (72, 3), (1028, 1), (2048, 16)])
def test_quads_are_the_single_channels_bits(W, blocks, lengths):
    g = torch.Generator().manual_seed(W)
    T, B, b = sum(lengths), len(lengths), W // blocks
    draw = lambda *shape: torch.randn(*shape, generator=g)
    proj, bx, by, taps, fb, conv = draw(T, 2 * W), draw(W), draw(W), draw(W, 4), draw(W), draw(B + 1, 3, W)
    gates, rb, ib, lam, state = draw(T, 2 * W), draw(W), draw(W), draw(W) * 3, draw(B + 1, W)
    starts = torch.tensor([0] + lengths).cumsum(0).to(torch.int32)
    seq_of = torch.cat([torch.full((n,), i, dtype=torch.int32) for i, n in enumerate(lengths)])
    meta = types.SimpleNamespace(max_new=max(lengths), num_seqs=B, num_tokens=T, seq_starts=starts.to(DEV), host_starts=starts.numpy(),
                                 seq_of=seq_of.to(DEV), slots=torch.arange(B, 0, -1, dtype=torch.int32, device=DEV), derived={})
    got = []
    for odd in (False, True):
        ug = placed(torch.zeros(T, 2 * W), odd)
        kept = conv.to(DEV)
        recurrent.lru_inputs(placed(proj, odd), bx.to(DEV), by.to(DEV), taps.to(DEV), fb.to(DEV), kept, meta, ug)
        pre, held = placed(gates, odd), state.to(DEV)
        out = torch.empty(T, W, device=DEV)
        recurrent.lru_scan(ug, pre, rb.to(DEV), ib.to(DEV), lam.to(DEV), 8.0, held, meta, out, b)
        got.append((ug.clone(), kept, pre.clone(), out, held))
    for one, other in zip(*got):
        assert torch.equal(one, other)
