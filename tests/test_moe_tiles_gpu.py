"""The experts' products by tall row tiles (csrc/moe.hip, grouped_tile_kernel): every height against float64."""
import pytest
import torch

from herbert_rs_amd.kernels import moe

DEV = "cuda"


@pytest.mark.gpu
@pytest.mark.parametrize("tile_m", moe.TALL_TILES)
@pytest.mark.parametrize("T,E,real,top,W,F", [(1, 2, 2, 1, 64, 64), (129, 1, 1, 1, 128, 64), (700, 3, 3, 2, 192, 128),
                                              (900, 5, 4, 2, 320, 448), (513, 2, 2, 1, 1024, 192)])
def test_tall_tiles(T, E, real, top, W, F, tile_m):
    """One row, rows that just pass a tile, experts with none, experts without matrices; one step of k and several; columns that
    fill no block of 256. The sums are float32 over bfloat16 operands: off by at most K roundings of the terms' sizes; the
    gated unit is rounded to bfloat16 (2^-9, and as much for what its inputs are off)."""
    g = torch.Generator().manual_seed(T + F)
    logits = torch.randn(T, E, generator=g)
    logits[:, 0] += 1.0                                     # (unequal experts)
    y = torch.randn(T, W, generator=g).bfloat16()
    gate_up = (torch.randn(real, 2 * F, W, generator=g) * W ** -0.5).bfloat16()
    down = (torch.randn(real, W, F, generator=g) * F ** -0.5).bfloat16()
    r = moe.Routing(torch.empty(moe.Routing.ints_needed(T, E, top, tile_m), dtype=torch.int32, device=DEV),
                    torch.empty(T, top, device=DEV), T, E, top, real=real, tall=tile_m)
    moe.route(logits.to(DEV), None, r)
    act = torch.full((T * top, F), 7.0, dtype=torch.bfloat16, device=DEV)
    out = torch.full((T * top, W), 7.0, device=DEV)
    moe.grouped_mfma(y.to(DEV), W, 0, moe.pack_grouped(gate_up).to(DEV), act, F, 0, moe.EPI_GLU, r, gather=True, limit=2.0, alpha=1.702,
                     tall=True)
    moe.grouped_mfma(act, F, 0, moe.pack_grouped(down).to(DEV), out, W, 0, moe.EPI_F32, r, tall=True)
    counts, tiles, row = r.counts.tolist(), [], 0
    for e, c in enumerate(counts):
        tiles += [(e if e < real else -1, row + i, min(tile_m, c - i)) for i in range(0, c, tile_m)]
        row += c
    got = list(zip(*r.tall_list.tolist()))
    assert got[:len(tiles)] == tiles and all(t[0] == -1 for t in got[len(tiles):])
    order, chosen = r.order.cpu().long(), r.chosen.cpu().long()
    expert = chosen[order]
    for e in range(E):
        rows = (expert == e).nonzero().flatten()
        if not rows.numel():
            continue
        if e >= real:                                       # no matrices: nothing is written
            assert bool((act[rows] == 7.0).all()) and bool((out[rows] == 7.0).all())
            continue
        x = y[order[rows] // top].double() @ gate_up[e].double().T
        gate, up = x[:, :F].clamp(max=2.0), x[:, F:].clamp(-2.0, 2.0)
        want = gate * torch.sigmoid(1.702 * gate) * (up + 1.0)
        got = act[rows].cpu().double()
        assert bool(((got - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all()), e
        terms = got @ down[e].double().T
        size = got.abs() @ down[e].double().abs().T
        assert bool(((out[rows].cpu().double() - terms).abs() <= F * 2.0 ** -24 * size + 1e-30).all()), e


@pytest.mark.gpu
@pytest.mark.parametrize("T,E,top,tall", [(1, 3, 2, 0), (8, 5, 3, 0), (8, 5, 3, 128), (9, 4, 1, 0), (70, 3, 2, 0), (300, 3, 2, 192), (257, 2, 1, 256)])
def test_rows_of_a_shared_expert(T, E, top, tall):
    """An expert that every token takes, its matrices behind the others': a row a token behind the pairs', its tiles behind
    theirs in either list; the pairs' own parts are what they are without it. Products and sum against float64 (bounds as above;
    the sum of top + 1 terms adds as many roundings)."""
    W, F = 128, 64
    g = torch.Generator().manual_seed(T)
    logits, y = torch.randn(T, E, generator=g).to(DEV), torch.randn(T, W, generator=g).bfloat16()
    gate = torch.randn(T, 3, generator=g).to(DEV)
    gate_up = (torch.randn(E + 1, 2 * F, W, generator=g) * W ** -0.5).bfloat16()
    down = (torch.randn(E + 1, W, F, generator=g) * F ** -0.5).bfloat16()
    made = {}
    for shared in (False, True):
        r = moe.Routing(torch.full((moe.Routing.ints_needed(T, E, top, tall, shared),), -7, dtype=torch.int32, device=DEV),
                        torch.empty(T, top, device=DEV), T, E, top, tall=tall, shared=shared)
        moe.route(logits, None, r)
        made[shared] = r
    r, A = made[True], T * top
    for name in ("chosen", "row_of", "counts", "weight"):
        assert torch.equal(getattr(r, name), getattr(made[False], name))
    assert torch.equal(r.order[:A], made[False].order) and torch.equal(r.order[A:].cpu(), torch.arange(T, dtype=torch.int32) * top)
    lists = [(64, torch.stack([r.tile_expert, r.tile_row0, r.tile_rows]))] + ([(tall, r.tall_list)] if tall else [])
    for rows, got in lists:
        want, at = [], 0
        for e, c in enumerate(r.counts.tolist() + [T]):
            want += [(e, at + i, min(rows, c - i)) for i in range(0, c, rows)]
            at += c
        got = list(zip(*got.tolist()))
        assert got[:len(want)] == want and all(t[0] == -1 for t in got[len(want):])
    act = torch.empty(r.rows, F, dtype=torch.bfloat16, device=DEV)
    out = torch.empty(r.rows, W, device=DEV)
    moe.grouped_mfma(y.to(DEV), W, 0, moe.pack_grouped(gate_up).to(DEV), act, F, 0, moe.EPI_GLU, r, gather=True, limit=float("inf"),
                     alpha=1.0, shift=0.0, tall=tall > 0)
    moe.grouped_mfma(act, F, 0, moe.pack_grouped(down).to(DEV), out, W, 0, moe.EPI_F32, r, tall=tall > 0)
    expert = torch.cat([r.chosen.cpu()[r.order.cpu().long()[:A]].long(), torch.full((T,), E)])
    got = act.cpu().double()
    for e in range(E + 1):
        rows = (expert == e).nonzero().flatten()
        x = y[r.order.cpu().long()[rows] // top].double() @ gate_up[e].double().T
        want = torch.nn.functional.silu(x[:, :F]) * x[:, F:]
        assert bool(((got[rows] - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all()), e
        size = got[rows].abs() @ down[e].double().abs().T
        assert bool(((out[rows].cpu().double() - got[rows] @ down[e].double().T).abs() <= F * 2.0 ** -24 * size + 1e-30).all()), e
    x = torch.zeros(T, W, device=DEV)
    moe.combine(out[:A], r, x, shared=out[A:], gate=(gate, 1))
    terms = out.cpu().double()[r.row_of.cpu().long()].view(T, top, W) * r.weight.cpu().double()[:, :, None]
    terms = torch.cat([terms, (torch.sigmoid(gate[:, 1:2].cpu().double()) * out[A:].cpu().double())[:, None]], 1)
    assert bool(((x.cpu().double() - terms.sum(1)).abs() <= (top + 4) * 2.0 ** -23 * terms.abs().sum(1) + 1e-30).all())


def test_tile_heights_by_the_rows_an_expert_has():
    """Few rows keep the low tiles, as do sizes that the tall ones refuse and steps that would leave most CUs without one."""
    assert moe.tall_rows(256, 4, 32, 32, 2048, 768) == 0
    assert moe.tall_rows(2048, 4, 32, 32, 2048, 800) == 0
    assert moe.tall_rows(1600, 2, 64, 64, 64, 64) == 0
    assert moe.tall_rows(768, 4, 32, 32, 2048, 768) == 128
    assert moe.tall_rows(1602, 4, 40, 32, 2048, 768) == 192
    assert moe.tall_rows(1712, 4, 32, 32, 2048, 768) == 256
    assert moe.tall_rows(1712, 4, 32, 32, 2048, 768, True) == 128
