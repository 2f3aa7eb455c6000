"""The latent attention of prompts that builds the heads' keys and values: against float64, at the edges of its tiles of 64
queries and 64 keys, with sequences that go on in the cache, sinks and gates, and keys that not every row sees; which sequences of
a step take this form, and steps whose sequences take one each."""
import numpy as np
import pytest
import torch

from herbert_rs_amd.cache import Cache, KVNeed
from herbert_rs_amd.kernels import latent, moe
from herbert_rs_amd.parts import PartSpec, Runtime, StepContext, build

from .test_vipalorn_kernels_gpu import DEV, rand, step_meta

pytestmark = pytest.mark.gpu


def setup(held, new, rank, rot):
    cache = Cache({0: KVNeed(1, rank + rot, None, values=False)}, 64 * sum(-(-n // 64) for n in held), 4096, torch.bfloat16, DEV,
                  max_slots=len(held))
    kv = cache.kv_view(0)
    slots = [cache.alloc_slot() for _ in held]
    for s, n, k in zip(slots, held, new):
        if n > k:
            step_meta(cache, [s], [n - k])
    meta = step_meta(cache, slots, new)
    kv.k.fill_(float("nan"))
    rows = [rand(n, rank + rot, seed=i).to(torch.bfloat16) for i, n in enumerate(held)]
    for s, r in zip(slots, rows):
        table = kv.page_table[s].cpu().tolist()
        for p in range(r.shape[0]):
            kv.k[table[p // 64], 0, p % 64] = r[p].to(DEV)
    return cache, kv, slots, meta, rows


@pytest.mark.parametrize("H,D,rank,rot", [(16, 128, 512, 64), (3, 128, 96, 0), (5, 64, 256, 32), (1, 64, 32, 64), (2, 128, 480, 32),
                                          (7, 64, 128, 0)])
def test_built_heads_against_float64(H, D, rank, rot):
    """Keys and values in bfloat16 (2^-9 of an entry each), queries and weights in 16 bits, an output of 8: 2^-8 of the largest
    entry for the output and values, and the scores' error (2^-9 of a key's entries, as independent errors over dim entries)
    times the spread of the values."""
    held, new = [150, 70, 1, 97, 64, 65, 300, 33], [150, 30, 1, 97, 64, 65, 129, 32]
    cache, kv, slots, meta, rows = setup(held, new, rank, rot)
    T, dims = sum(new), D + rot
    uk, uv = (rand(H, D, rank, seed=20 + i, scale=rank ** -0.5).to(torch.bfloat16) for i in (0, 1))
    q, turned, gate, sinks = rand(T, 5 + H * dims, seed=9), rand(T, H * rot, seed=12), rand(T, H + 1, seed=10), rand(H, seed=11)
    scale, buffer = 2.0 * dims ** -0.5, Runtime(torch.bfloat16, DEV).buffer

    def run():
        out = torch.empty(T, H * D, dtype=torch.bfloat16, device=DEV)
        latent.latent_attention_heads(q.to(DEV), 5, turned.to(DEV), meta, kv, moe.pack_grouped(uk.to(DEV)), moe.pack_grouped(uv.to(DEV)),
                                      out, gate.to(DEV), 1, D, D, rank, rot, scale, buffer, sinks=sinks.to(DEV))
        return out.cpu()
    out, at = run(), 0
    for r, n, k in zip(rows, held, new):
        r = r.double()
        keys = torch.cat([torch.einsum("tr,hdr->htd", r[:, :rank], uk.double()), r[:, rank:].expand(H, -1, -1)], -1)
        values = torch.einsum("tr,hdr->htd", r[:, :rank], uv.double())
        query = torch.cat([q[at:at + k, 5:].view(k, H, dims)[..., :D], turned[at:at + k].view(k, H, rot)], -1).double().transpose(0, 1)
        score = query @ keys.transpose(1, 2) * scale
        see = torch.arange(n)[None, :] <= torch.arange(n - k, n)[:, None]
        score = torch.cat([score.masked_fill(~see, -torch.inf), sinks.double()[:, None, None].expand(H, k, 1)], -1)
        want = torch.softmax(score, -1)[..., :-1] @ values * torch.sigmoid(gate[at:at + k, 1:].double()).T[..., None]
        got = out[at:at + k].view(k, H, D).transpose(0, 1).double()
        # the largest of some 10^5 errors of that deviation: five of them
        spread = float(scale * (query.norm(dim=-1)).max() * 2.0 ** -9 / 3 ** 0.5)
        bound = (2.0 ** -8 + 5 * spread * 2.0 ** -2) * float(values.abs().max())
        assert float((got - want).abs().max()) <= bound, (n, k)
        assert float((got - want).norm() / want.norm()) <= 2.0 ** -7, (n, k)
        at += k
    # a later token's row without finite numbers, and one that is only larger: the tokens before it are the same bits
    late, table = 140, kv.page_table[slots[0]].cpu().tolist()
    for what in (float("inf"), float("nan"), 40.0):
        kv.k[table[late // 64], 0, late % 64, 7:9] = what
        again = run()
        assert torch.equal(again[:late], out[:late]) and torch.equal(again[150:], out[150:])
        assert not torch.equal(again[late:150], out[late:150])
        if what != 40.0:
            assert not again[late:150].isfinite().any()


def test_a_sequence_is_the_same_bits_alone():
    """A row's sums run over blocks of keys at absolute positions: alone or beside others, the same bits."""
    H, D, rank, rot, held = 4, 128, 128, 64, [200, 90, 131]
    cache, kv, slots, meta, rows = setup(held, held, rank, rot)
    uk, uv = (moe.pack_grouped(rand(H, D, rank, seed=20 + i, scale=rank ** -0.5).to(torch.bfloat16).to(DEV)) for i in (0, 1))
    q, turned = rand(sum(held), H * (D + rot), seed=9).to(DEV), rand(sum(held), H * rot, seed=12).to(DEV)
    out = torch.empty(sum(held), H * D, dtype=torch.bfloat16, device=DEV)
    buffer = Runtime(torch.bfloat16, DEV).buffer
    latent.latent_attention_heads(q, 0, turned, meta, kv, uk, uv, out, None, 0, D, D, rank, rot, 0.1, buffer)
    for i, n in enumerate(held):
        first = sum(held[:i])
        one, kv1, _, meta1, _ = setup([n], [n], rank, rot)
        table, table1 = kv.page_table[slots[i]].cpu().tolist(), kv1.page_table[0].cpu().tolist()
        for p in range(n):
            kv1.k[table1[p // 64], 0, p % 64] = rows[i][p].to(DEV)
        alone = torch.empty(n, H * D, dtype=torch.bfloat16, device=DEV)
        latent.latent_attention_heads(q[first:first + n].contiguous(), 0, turned[first:first + n].contiguous(), meta1, kv1, uk, uv,
                                      alone, None, 0, D, D, rank, rot, 0.1, buffer)
        assert torch.equal(alone, out[first:first + n]), i


def test_the_line_between_the_forms():
    """Prompts and portions build the heads, short prompts too (whatever is beside them); single tokens, a few tokens each of many
    long sequences and sizes that the kernels do not take do not."""
    kv = type("KV", (), {"k": torch.empty(0, dtype=torch.bfloat16), "page_size": 64})

    def pays(context, new, H=16, dim=128, vdim=128, rank=512, rot=64):
        meta = type("Meta", (), {"max_new": max(new), "max_context": max(context), "host_context": np.array(context, dtype=np.int32),
                                 "host_starts": np.concatenate([[0], np.cumsum(new)]).astype(np.int32)})
        return latent.heads_pay(meta, kv, H, dim, vdim, rank, rot)
    assert pays([2048], [2048]) and pays([1400, 900], [1400, 900]) and pays([8192], [512]) and pays([8192], [20])
    assert not pays([2048], [1]) and pays([64], [64]) and not pays([4096] * 32, [4] * 32)
    assert not pays([200000], [512])                    # scratch
    assert not pays([2048], [2048], vdim=64) and not pays([2048], [2048], dim=96, vdim=96) and not pays([2048], [2048], rot=128)


def test_more_sequences_than_a_wave_looks_at_a_time():
    """130 sequences of unequal lengths, some without tiles of their own in the list: the tiles of the 64th, 65th and 129th follow
    those before them. Every sequence is the same bits as in a call that names it alone, and so is a list of some in another order."""
    H, D, rank, rot = 2, 64, 64, 32
    new = [2 + (37 * i) % 97 for i in range(130)]
    held = [n + (70 if i % 7 == 3 else 0) for i, n in enumerate(new)]
    cache, kv, slots, meta, rows = setup(held, new, rank, rot)
    uk, uv = (moe.pack_grouped(rand(H, D, rank, seed=20 + i, scale=rank ** -0.5).to(torch.bfloat16).to(DEV)) for i in (0, 1))
    q, turned = rand(sum(new), H * (D + rot), seed=9).to(DEV), rand(sum(new), H * rot, seed=12).to(DEV)
    buffer = Runtime(torch.bfloat16, DEV).buffer

    def run(names=None):
        out = torch.full((sum(new), H * D), 7.0, dtype=torch.bfloat16, device=DEV)
        call = None
        if names is not None:
            call = (torch.tensor(names, dtype=torch.int32, device=DEV), len(names), sum(-(-held[i] // 64) for i in names), max(new[i] for i in names))
        latent.latent_attention_heads(q, 0, turned, meta, kv, uk, uv, out, None, 0, D, D, rank, rot, 0.2, buffer, call=call)
        return out
    whole, starts = run(), np.concatenate([[0], np.cumsum(new)])
    for i in [0, 1, 62, 63, 64, 65, 127, 128, 129]:
        one = run([i])
        assert torch.equal(one[starts[i]:starts[i + 1]], whole[starts[i]:starts[i + 1]]), i
        assert bool((one[:starts[i]] == 7.0).all()) and bool((one[starts[i + 1]:] == 7.0).all()), i
    some = [i for i in range(129, -1, -1) if i % 3]
    listed = run(some)
    for i in range(130):
        want = whole[starts[i]:starts[i + 1]] if i in some else torch.full_like(whole[starts[i]:starts[i + 1]], 7.0)
        assert torch.equal(listed[starts[i]:starts[i + 1]], want), i


@pytest.mark.parametrize("q_rank,gate", [(None, True), (64, False)])
@pytest.mark.parametrize("held,new", [([300, 40, 900, 130, 5], [1, 40, 1, 130, 5]), ([200, 200, 200, 300], [1, 1, 1, 300]), ([64, 700, 120], [64, 3, 120]),
                                      ([90, 4000], [90, 2]), ([150, 70] * 5, [1, 70, 3, 64, 1, 70, 1, 70, 2, 70])])
def test_the_same_rows_through_both_forms(held, new, q_rank, gate, monkeypatch):
    """A layer's step with a form a sequence, against all of them scoring on the latents and all of them built (single tokens too). Five
    kinds of numbers are rounded to bfloat16 in either form (queries or mapped queries, keys or latents, values or summed latents, the
    outputs, the output product's rows), each by up to 2^-9 of itself: 2^-7 of a sequence's norm between any two."""
    H, D, rank, rot, W = 4, 64, 128, 32, 192
    position = PartSpec("rope", {"theta": 500.0, "rotary_dims": rot, "max_positions": 8192, "tables": False})
    names = {n: n for n in ("dkv", "dkv_norm", "uk", "uv", "o")} | ({"dq": "dq", "dq_norm": "dq_norm", "uq": "uq"} if q_rank else {"q": "q"})
    names["g"] = "g" if gate else None
    part = build("mixer", PartSpec("latent_attention", {
        "hidden_size": W, "heads": H, "dim": D, "rot_dim": rot, "vdim": D, "kv_rank": rank, "scale": (D + rot) ** -0.5, "eps": 1e-6,
        "position": position, "names": names, "q_rank": q_rank}),
        shared=type("Shared", (), {"position": staticmethod(lambda spec: build("position", spec))}))
    rt = Runtime(torch.bfloat16, DEV)
    part.position.load({}, rt)
    part.load({n: (1 + 0.1 * rand(*need.shape, seed=i) if need.role == "scale" else rand(*need.shape, seed=i, scale=need.shape[-1] ** -0.5).to(torch.bfloat16))
               for i, (n, need) in enumerate(sorted(part.tensor_needs().items()))}, rt)
    y = rand(sum(new), W, seed=3).to(torch.bfloat16).to(DEV)
    choice, got = latent._sequence_form, {}
    for name in ("own", "latents", "built"):
        monkeypatch.setattr(latent, "_sequence_form", lambda *a: choice(*a) if name == "own" else (name == "built",) + choice(*a)[1:])
        cache, kv, slots, meta, rows = setup(held, new, rank, rot)
        kv.k.nan_to_num_(0.0)                               # (what the step itself writes is not there yet)
        x = torch.zeros(sum(new), W, device=DEV)
        ctx = StepContext(rt=rt, meta=meta, cache=cache)
        part.forward(ctx, y, x)
        if name == "own":
            forms = latent.forms(meta, kv, H, D, D, rank, rot)
            assert forms.calls and forms.rest
        got[name] = x.cpu().double()
    at = 0
    for n in new:
        for a, b in (("own", "latents"), ("own", "built"), ("built", "latents")):
            one, other = got[a][at:at + n], got[b][at:at + n]
            assert float((one - other).norm() / other.norm()) <= 2.0 ** -7, (a, b, n)
        at += n
