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
    # (the low ones where the tall ones would take a round more than they save)
    assert moe.tall_rows(800, 4, 64, 64, 4096, 1536, True) == 0 and moe.tall_rows(1500, 4, 64, 64, 4096, 1536, True) == 128
    assert moe.tall_rows(512, 6, 64, 64, 2048, 1408, True) == 0 and moe.tall_rows(1600, 8, 256, 256, 2048, 512) == 0


def test_tiles_of_the_down_product():
    """Tall tiles where their rounds are done sooner than the low tiles': both sides of the lines in steps of k, rows and rounds."""
    assert not moe.down_tall(2048, 4, 32, 32, 2048, 768, False, 0)
    assert moe.down_tall(2048, 4, 32, 32, 2048, 768, False, 128) and not moe.down_tall(2048, 4, 32, 32, 2048, 704, False, 128)
    assert not moe.down_tall(2048, 4, 32, 32, 2048, 768, True, 192)
    assert moe.down_tall(1712, 4, 32, 32, 2048, 768, False, 256) and not moe.down_tall(1000, 4, 32, 32, 2048, 768, False, 128)
    assert moe.down_tall(2500, 4, 64, 64, 4096, 1536, False, 192) and not moe.down_tall(1500, 4, 64, 64, 4096, 1536, False, 128)


def test_down_products_of_16_steps_and_more_take_the_tall_tiles():
    """From 128 rows an expert on whatever the rounds, which the estimate counts too high where experts are about as busy as the mean."""
    assert moe.down_tall(1400, 6, 64, 64, 2048, 1408, False, 192) and moe.down_tall(700, 2, 8, 8, 4096, 3584, False, 256)
    assert moe.down_tall(1400, 6, 64, 64, 2048, 1024, False, 192) and not moe.down_tall(1400, 6, 64, 64, 2048, 960, False, 192)
    assert not moe.down_tall(1300, 6, 64, 64, 2048, 1408, False, 192) and not moe.down_tall(1400, 6, 64, 64, 2048, 1408, False, 0)


def test_a_shared_expert_is_folded_only_where_that_pays():
    """Both sides of the lines: always beyond the steps of few rows an expert, in them while its rows are few tiles of matrices
    that are small enough to be read again."""
    assert all(moe.fold_pays(T, 4, 32, 2048, 768) for T in (1, 8, 128, 129, 512, 2048, 8192))
    assert all(moe.fold_pays(T, 8, 256, 2048, 512) for T in (1, 64, 512, 513, 2048))
    assert moe.fold_pays(512, 1, 128, 2048, 768) and not moe.fold_pays(1024, 1, 128, 2048, 768)
    assert not moe.fold_pays(2048, 1, 128, 2048, 768) and moe.fold_pays(2049, 1, 128, 2048, 768)
    assert moe.fold_pays(32, 4, 64, 4096, 1536) and not moe.fold_pays(33, 4, 64, 4096, 1536)
    assert not moe.fold_pays(256, 4, 64, 4096, 1536) and moe.fold_pays(257, 4, 64, 4096, 1536)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [1, 7, 70, 300])
def test_a_shared_expert_folded_and_by_its_own_products(T, monkeypatch):
    """The same layer either way. The shared expert's activations are rounded to bfloat16 from float32 sums in another order, so one may
    fall to the neighbouring value (2^-7 of it); its product passes that on, the sums themselves are off by K roundings."""
    from herbert_rs_amd.parts import PartSpec, Runtime, StepContext, build
    E, top, W, F = 6, 2, 128, 64
    part = build("feed_forward", PartSpec("routed_experts", {
        "hidden_size": W, "intermediate_size": F, "experts": E, "top": top, "activation": "silu", "routing": "scores",
        "names": {"router": "r", "router_bias": "b", "gate": "g{e}", "up": "u{e}", "down": "d{e}"},
        "shared_expert": {"intermediate_size": F, "names": {"gate": "sg", "up": "su", "down": "sd", "sg": "s"}}}))
    g = torch.Generator().manual_seed(T)
    tensors = {name: torch.randn(*need.shape, generator=g) * need.shape[-1] ** -0.5 for name, need in part.tensor_needs().items()}
    rt = Runtime(torch.bfloat16, DEV)
    part.load({name: t if name == "b" else t.bfloat16() for name, t in tensors.items()}, rt)
    assert part.foldable
    y, got = torch.randn(T, W, generator=g).bfloat16(), {}
    for fold in (False, True):
        monkeypatch.setattr(moe, "fold_pays", lambda *a: fold)
        got[fold] = torch.zeros(T, W, device=DEV)
        part.forward(StepContext(rt=rt, meta=None, cache=None), y.to(DEV), got[fold])
    x = y.double()
    gate, up, down, sg = (tensors[n].bfloat16().double() for n in ("sg", "su", "sd", "s"))
    act = torch.nn.functional.silu(x @ gate.T) * (x @ up.T)
    size = torch.sigmoid(x @ sg.T) * (act.abs() @ down.abs().T)
    off = (got[True] - got[False]).cpu().double().abs()
    assert bool((off <= 2.0 ** -7 * size + 2.0 ** -20 * (got[False].cpu().double().abs() + size)).all())
    assert float(size.min()) > 0 and bool((got[True].cpu().double().abs().sum(1) > 0).all())


@pytest.mark.gpu
def test_rows_by_tall_tiles_and_by_low_ones():
    """The same rows by tiles of 64 and by every tall height: k is added in another order, so the float32 sums differ by
    at most K roundings of the terms' sizes either way; the heights agree bit for bit."""
    T, E, top, W, F = 700, 3, 2, 256, 128
    g = torch.Generator().manual_seed(3)
    logits, y = torch.randn(T, E, generator=g).to(DEV), torch.randn(T, W, generator=g).bfloat16()
    w = (torch.randn(E, F, W, generator=g) * W ** -0.5).bfloat16()
    got = {}
    for height in (0,) + moe.TALL_TILES:
        r = moe.Routing(torch.empty(moe.Routing.ints_needed(T, E, top, height), dtype=torch.int32, device=DEV),
                        torch.empty(T, top, device=DEV), T, E, top, tall=height)
        moe.route(logits, None, r)
        got[height] = torch.empty(T * top, F, device=DEV)
        moe.grouped_mfma(y.to(DEV), W, 0, moe.pack_grouped(w).to(DEV), got[height], F, 0, moe.EPI_F32, r, gather=True, tall=height > 0)
    order, chosen = r.order.cpu().long(), r.chosen.cpu().long()
    rows, expert = y[order // top].double(), chosen[order]
    size = torch.stack([rows[i].abs() @ w[expert[i]].double().abs().T for i in range(T * top)])
    assert torch.equal(got[128], got[192]) and torch.equal(got[128], got[256])
    off = (got[128].cpu().double() - got[0].cpu().double()).abs()
    assert bool((off <= 2 * W * 2.0 ** -24 * size).all())
