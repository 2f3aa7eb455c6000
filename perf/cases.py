"""What this library is timed on: passes of whole models through its step function.

A case is a model of one of the seven designs at one of the sizes that bench.py uses, a compute type, a
batch of sequences and what is asked of them:

  prompt   the prompts of a batch go through in one step, each sequence's last logits are wanted; the
           sequences are given back (a request's first token, a document that is scored)
  serve    the same, then `new` decode steps of the whole batch (whole requests, start to end)
  decode   one decode step of sequences that hold `prompt` tokens already (the long middle of a
           generation), then rolled back by that token so that every pass is the same step; for the
           dense decoder only, whose cache can be rolled back

Tokens are given, as trace replay and scoring give them, so that a pass does not depend on near-ties of
its own logits. Weights are random with the deviations that random models of this library have, so
that no mechanism is idle, but for two things that keep bfloat16's rounding from deciding what comes
out, as it does not in a trained model: the embedding is as large as what dozens of layers add to it, and
routers read signs that no layer writes over (see `weight`). `exact` says what the same passes give in 64 bits: plain whole-sequence formulas
without a cache.
"""
import functools
import math
import zlib

import torch

import herbert_rs_amd as hb
from herbert_rs_amd.config.registry import resolve_architecture
from herbert_rs_amd.engine import StepEntry
from herbert_rs_amd.engine.model import Model

VOCAB = 32768
# width, layers, heads, key dim, value dim, latent rank, rotated part, experts, top, expert width
SIZES = {"small": (1024, 4, 8, 128, 128, 256, 64, 16, 2, 512),
         "medium": (2048, 8, 16, 128, 128, 512, 64, 32, 4, 768),
         "wide": (4096, 4, 32, 128, 128, 512, 64, 64, 4, 1536)}
# layers, width, query heads, kv heads, feed-forward, vocabulary, tied embedding: the shapes of BASELINE.md's decoder
DENSE = {"8b": (36, 4096, 32, 8, 12288, 151936, False), "1.7b": (28, 2048, 16, 8, 6144, 151936, True)}
FAMILIES = ("qwen3", "vipalorn", "modasun", "mefatar", "bozasun", "mutedra", "figalorn")


# ---------------------------------------------------------------- the cases
def case(name, family, size, what, batch, prompt, spread=0.0, new=0, dtype="bfloat16"):
    return {"name": name, "family": family, "size": size, "what": what, "batch": batch, "prompt": prompt,
            "spread": spread, "new": new, "dtype": dtype}


def listed():
    return [
        # one user's next token on a small model: nothing but latency and launches
        case("next_token_small", "qwen3", "small", "decode", 1, 100),
        # eight users' next tokens on the 8B shape at 4,096 tokens each: the library's headline
        case("decode_8b_batch8", "qwen3", "8b", "decode", 8, 4095),
        # one user's prompt on the 8B shape: time to the first token
        case("prompt_8b", "qwen3", "8b", "prompt", 1, 2048),
        # sixteen requests of unequal lengths that arrive together, 1.7B shape
        case("requests_1.7b", "qwen3", "1.7b", "prompt", 16, 1024, spread=0.9),
        # many users of unequal contexts, 1.7B shape
        case("decode_1.7b_batch48", "qwen3", "1.7b", "decode", 48, 1500, spread=0.6),
        # the all-float32 mode, as used to check a model's numbers: a prompt and a few tokens
        case("float32_requests", "qwen3", "medium", "serve", 2, 333, spread=0.5, new=4, dtype="float32"),
        # a long prompt through delta layers, latent attention and routed experts
        case("prompt_vipalorn", "vipalorn", "medium", "prompt", 1, 2048),
        # short requests served whole by channel-decay delta layers and grouped experts
        case("requests_modasun", "modasun", "medium", "serve", 8, 301, spread=0.7, new=8),
        # a prompt of odd length through recurrent units and two mixers side by side
        case("prompt_mefatar", "mefatar", "medium", "prompt", 1, 1777),
        # requests through state-space layers, chunked and latent attention, experts with identities
        case("requests_bozasun", "bozasun", "medium", "serve", 4, 509, spread=0.5, new=8),
        # three documents beyond the window, layers that run twice
        case("documents_mutedra", "mutedra", "medium", "prompt", 3, 1400, spread=0.4),
        # a wide batch of short requests through difference maps and key-valued windows
        case("requests_figalorn", "figalorn", "wide", "serve", 24, 90, spread=0.8, new=8),
    ]


def draw(rng):
    """Any family and kind of pass, the sizes over their logarithm; the largest cost what `prompt_8b` costs or less."""
    family = rng.choice(FAMILIES + ("qwen3", "qwen3"))
    dtype = "float32" if rng.random() < 0.12 else "bfloat16"
    size = rng.choice(("small", "medium", "medium", "wide")
                      + (("1.7b", "1.7b") if family == "qwen3" and dtype == "bfloat16" else ()))
    what = rng.choice(("prompt", "serve", "decode") if family == "qwen3" else ("prompt", "serve"))
    most = 300 if dtype == "float32" else {"decode": 30000, "prompt": 4000, "serve": 2000}[what]
    batch = int(round(math.exp(rng.uniform(0.0, math.log(48.0 if dtype == "bfloat16" else 8.0)))))
    top = max(8, min(most // batch, 4000))
    prompt = int(round(math.exp(rng.uniform(math.log(6.0), math.log(top)))))
    spread = rng.choice((0.0, 0.3, 0.6, 0.9)) if batch > 1 else 0.0
    return {"family": family, "size": size, "what": what, "batch": batch, "prompt": prompt, "spread": spread,
            "new": rng.randint(2, 4 if dtype == "float32" else 10) if what == "serve" else 0, "dtype": dtype}


def lengths(c):
    """Prompt lengths: the first sequence's is the longest, the others' lie anywhere down to (1 - spread) of it. (A step
    that starts a new page of the cache is one in 64: no decode case is made of those.)"""
    out = [max(1, int(round(c["prompt"] * (1.0 - c["spread"] * ((i * 0.6180339887) % 1.0))))) for i in range(c["batch"])]
    return [n + 1 if c["what"] == "decode" and n % 64 == 0 else n for n in out]


# ---------------------------------------------------------------- configurations
def config(c):
    family = c["family"]
    if family == "qwen3":
        if c["size"] in DENSE:
            L, W, H, G, ff, vocab, tied = DENSE[c["size"]]
        else:
            W, L, H, _, _, _, _, _, top, eff = SIZES[c["size"]]
            G, ff, vocab, tied = H // 2, top * eff, VOCAB, True
        return dict(architectures=["Qwen3ForCausalLM"], model_type="qwen3", num_hidden_layers=L, hidden_size=W,
                    num_attention_heads=H, num_key_value_heads=G, head_dim=128, intermediate_size=ff,
                    vocab_size=vocab, rope_theta=1e6, rms_norm_eps=1e-6, tie_word_embeddings=tied,
                    max_position_embeddings=8192, eos_token_id=1)
    W, L, H, D, V, rank, R, E, top, ff = SIZES[c["size"]]
    dense = {"kind": "dense", "ff": top * ff}
    latent = {"heads": H, "dim": D, "rot_dim": R, "vdim": V, "kv_rank": rank, "scale": (D + R) ** -0.5,
              "rot": {"base": 10000.0, "dims": R}}
    heads = {"heads": H, "kv_heads": H // 2, "dim": D, "vdim": V, "scale": D ** -0.5}
    rows = {"heads": H, "kv_heads": H // 2, "dim": D, "vdim": V, "conv": 4}

    def build(kinds, runs, mlp=None):
        return [dict({"type": kinds[i % len(kinds)][0], "mixer": kinds[i % len(kinds)][1], "mlp": mlp}) for i in range(runs)]

    if family == "vipalorn":
        mlp = {"kind": "moe", "expert": {"ff": ff, "limit": 7.0}, "router": {"experts": E, "top": top}}
        return {"architecture": "Vipalorn", "vocab": VOCAB, "width": W, "norm": {"eps": 1e-5}, "residual_mult": 0.5,
                "logit_scale": 1.0, "layers": build([("delta", rows)] * 3 + [("latent_attention", latent)], L, mlp)}
    if family == "modasun":
        delta = dict(rows, low_rank={"decay": W // 16, "gate": W // 16})
        attention = dict(heads, q_temp={"coef": 0.1, "every": 1024})
        mlp = {"kind": "moe", "expert": {"ff": ff}, "shared": {"ff": ff},
               "router": {"experts": E, "top": top, "groups": {"count": 4, "keep": 2}}}
        return {"architecture": "Modasun", "vocab": VOCAB, "width": W, "norm": {"eps": 1e-5}, "postln_alpha": 2.0,
                "embedding": {"scale": 8.0}, "layers": build([("channel_delta", delta)] * 3 + [("attention", attention)], L, mlp)}
    if family == "mefatar":
        scaling = {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}
        left = dict(heads, conv=4, rot={"dims": D, "base": 10000.0, "scaling": scaling})
        right = {"heads": H // 2, "dim": D // 2, "vdim": V, "tau": 16.0, "rank": W // 16}
        kinds = [("rglru", {"width": W, "blocks": H, "conv": 4})] * 2 + [("parallel", {"left": left, "right": right})]
        return {"architecture": "Mefatar", "vocab": VOCAB, "width": W, "norm": {"eps": 1e-6}, "layers": build(kinds, L, dense)}
    if family == "bozasun":
        mlp = {"kind": "moe", "expert": {"ff": ff}, "router": {"experts": E, "top": top, "identity": E // 4,
                                                               "groups": {"count": 4, "keep": 2}}}
        space = {"heads": 2 * W // 64, "vdim": 64, "state": 128, "groups": 8, "conv": 4, "norm_groups": 8}
        attention = dict(heads, rot={"dims": D, "base": 1000000.0, "scaling": {"factor": 4.0}}, mask={"size": 2048}, softcap=50.0)
        kinds = [("mamba2", space), ("attention", attention), ("mamba2", space), ("latent_attention", latent)]
        return {"architecture": "Bozasun", "vocab": VOCAB, "width": W, "norm": {"eps": 1e-6}, "token_side": {"dim": 256},
                "layers": build(kinds, L, mlp)}
    if family == "mutedra":
        plain = {"heads": H, "dim": D, "vdim": V, "kv_rank": rank, "q_rank": W // 4, "scale": D ** -0.5}
        attention = dict(heads, bias_max=2560, mask={"size": 1024, "keep_first": 4})
        turned = ("latent_attention_2", dict(latent, q_rank=W // 4))
        kinds = [turned, ("attention", attention), ("latent_attention", plain), ("attention", attention), turned,
                 ("attention", attention)]
        return {"architecture": "Mutedra", "vocab": VOCAB, "width": W, "norm": {"eps": 1e-5}, "embedding": {"scale": 1.0},
                "loop": {"start": 0, "stop": 2, "times": 2}, "logit_softcap": 30.0, "layers": build(kinds, L - 2, dense)}
    window = dict(heads, softcap=50.0, mask={"size": 1024},
                  rot={"base": 10000.0, "dims": D, "scaling": {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}})
    maps = dict(heads, dim=D // 2, scale=(D // 2) ** -0.5, diff=0.5, mask={"size": 2048},
                rot={"base": 10000.0, "dims": D // 8, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}})
    return {"architecture": "Figalorn", "vocab": VOCAB, "width": W, "norm": {"eps": 1e-5},
            "loop": {"start": 0, "stop": 2, "times": 2},
            "layers": build([("attention_2", window), ("attention", maps)], L - 2, {"kind": "dense", "ff": 3 * top * ff // 2})}


def typed(raw):
    arch = resolve_architecture(raw)
    cfg = arch.config_class.from_dict(raw)
    return arch, cfg, arch.build_spec(cfg)


# ---------------------------------------------------------------- weights and tokens, from the seed alone
def spread_of(name, shape, family, width):
    """(mean, deviation) of a stored tensor: what this library's own random models have."""
    last = name.rsplit(".", 1)[-1]
    if last == "conv":
        return 1.0 / shape[1], 0.3
    if last in ("A_log", "dt_bias"):
        return 0.0, 0.5
    if last == "D":
        return 1.0, 0.3
    if last == "lam":
        return -2.2, 1.0
    if last == "alpha":
        return 0.7, 0.05
    if name.endswith("a2.b"):
        return 2.0, 1.0
    if last in ("lq1", "lk1", "lq2", "lk2"):
        return 0.0, 0.4 / shape[0] ** 0.25
    if last in ("sink", "rel"):
        return 0.0, 1.0
    if last in ("a2", "g2"):
        return 0.0, (2.0 / (0.02 * width ** 0.5) if family == "mefatar" else 1.0) / shape[1] ** 0.5
    if last in ("ra", "ri"):
        return 0.0, shape[-1] ** -0.5
    if last in ("b", "correction") and "mix.b" not in name or name == "loop.step":
        return 0.0, 0.002 if last == "correction" else 0.1 if "norm" in name or "mlp" in name else 0.4
    if last == "router":
        return 0.0, 0.02 if family == "modasun" else 0.1
    if name == "model.embed_tokens.weight":
        return 0.0, 1.0
    if "norm" in last or last in ("ls1", "ls2", "out") or name.endswith(("norm.weight", "layernorm.weight")):
        around_zero = family in ("modasun", "figalorn") and (last in ("norm1", "norm2") or name == "final.norm")
        return 0.0 if around_zero else 1.0, 0.1
    return 0.0, 0.02


ROUTED = ("vipalorn", "modasun", "bozasun")
SIGNS = 64


def weight(name, shape, c, seed, width):
    """A stored tensor. In the routed designs the first SIGNS channels of the residual stream hold signs of the token's
    own, the next SIGNS their opposites; norms scale both alike, no layer adds to either, and the routers
    read the differences: which experts a token takes varies from token to token and layer to layer, and does
    not hang on the last bit of a bfloat16 row."""
    if name.endswith(".rel"):
        shape = (32, shape[1])
    mean, deviation = spread_of(name, shape, c["family"], width)
    gen = torch.Generator(device="cuda").manual_seed(zlib.crc32(name.encode()) * 1000003 + int(seed))
    dtype = getattr(torch, c["dtype"])
    t = torch.randn(shape, generator=gen, device="cuda", dtype=dtype if mean == 0.0 else torch.float32)
    t = t.mul_(deviation).add_(mean).to(dtype) if mean else t.mul_(deviation)
    if c["family"] in ROUTED:
        first, both = slice(0, SIGNS), slice(0, 2 * SIGNS)
        after, last = slice(SIGNS, 2 * SIGNS), name.rsplit(".", 1)[-1]
        if name == "embed":
            t[:, first] = torch.where(t[:, first] < 0, -deviation, deviation).to(dtype)
            t[:, after] = -t[:, first]
        elif last == "router":
            t[:, after] = -t[:, first]
            t[:, 2 * SIGNS:] = 0
        elif name in ("embed.norm", "final.norm") or last in ("norm1", "norm2"):
            t[both] = mean
        elif last in ("o", "down", "proj") or name.endswith("mix.o.b"):
            t[both] = 0
    return t


def tokens(c, seed):
    """(prompts, decode steps' tokens [new or 1][batch]) as lists of ids."""
    gen = torch.Generator().manual_seed(int(seed) * 7919 + 11)
    vocab = DENSE[c["size"]][5] if c["size"] in DENSE else VOCAB
    prompts = [torch.randint(0, vocab, (n,), generator=gen).tolist() for n in lengths(c)]
    steps = torch.randint(0, vocab, (1 if c["what"] == "decode" else c["new"], c["batch"]), generator=gen).tolist()
    return prompts, steps


# ---------------------------------------------------------------- the passes
def prepare(c, seed):
    raw = config(c)
    arch, cfg, spec = typed(raw)
    width = raw.get("width", raw.get("hidden_size"))
    held = {name: weight(name, tuple(need.shape), c, seed, width) for name, need in Model(spec).tensor_needs().items()}
    room = sum((n + c["new"] + 129) // 64 * 64 for n in lengths(c))
    engine = hb.Engine(cfg, spec, held, dtype=c["dtype"], max_tokens=room, max_slots=c["batch"])
    prompts, steps = tokens(c, seed)
    state = {"engine": engine, "prompts": prompts, "steps": steps, "what": c["what"]}
    if c["what"] == "decode":
        slots = [engine.alloc_slot() for _ in prompts]
        for slot, p in zip(slots, prompts):
            engine.step([StepEntry(slot, p, [])])
        state["slots"] = slots
        for _ in range(2):          # a program that has been decoding: its steps are recorded
            run(state)
    return state


def run(state):
    engine, prompts, steps = state["engine"], state["prompts"], state["steps"]
    if state["what"] == "decode":
        logits = engine.step([StepEntry(s, [t], [0]) for s, t in zip(state["slots"], steps[0])])
        for s, p in zip(state["slots"], prompts):
            engine.truncate(s, len(p))
        return {"first": logits[:1], "rest": logits[1:]}
    slots = [engine.alloc_slot() for _ in prompts]
    out = [engine.step([StepEntry(s, p, [len(p) - 1]) for s, p in zip(slots, prompts)])]
    for ids in steps:
        out.append(engine.step([StepEntry(s, [t], [0]) for s, t in zip(slots, ids)]))
    for s in slots:
        engine.free_slot(s)
    return out


# ---------------------------------------------------------------- what a pass cannot do without
def visible_keys(m, n):
    """Keys that the query at position n sees."""
    mask = m.get("mask")
    if not mask:
        return n + 1
    if "bias_max" in m or "softcap" in m and "vdim" in m and mask["size"] == 1024:
        return min(n + 1, mask["size"] + mask.get("keep_first", 0))
    return n % mask["size"] + 1


def work(c):
    raw = config(c)
    spec = typed(raw)[2]
    model = Model(spec)
    elem = 4 if c["dtype"] == "float32" else 2
    W = raw.get("width", raw.get("hidden_size"))
    dense = expert = table = head = 0
    looped = raw.get("loop") or {"start": 0, "stop": 0, "times": 1}
    passes = 0                                  # weights that work a second time in the same step
    for name, need in model.tensor_needs().items():
        n = math.prod(32 if d is None else d for d in need.shape)
        if name in ("head", "lm_head.weight"):
            head += n
        elif "embed" in name and len(need.shape) == 2:
            table += n
            if name in ("embed", "model.embed_tokens.weight") and not {"head", "lm_head.weight"} & set(model.tensor_needs()):
                head += n
        elif ".mlp.e" in name:
            expert += n
        else:
            dense += n
            if name.startswith("l") and name[1].isdigit() and looped["start"] <= int(name[1:name.index(".")]) < looped["stop"]:
                passes += n * (looped["times"] - 1)
    layers = raw["layers"] if "layers" in raw else [{"type": "attention", "mixer": {
        "heads": raw["num_attention_heads"], "kv_heads": raw["num_key_value_heads"], "dim": 128, "vdim": 128}}] * raw["num_hidden_layers"]
    runs = list(range(looped["start"])) + list(range(looped["start"], looped["stop"])) * looped["times"] \
        + list(range(looped["stop"], len(layers)))
    routed = next((x["mlp"] for x in layers if (x.get("mlp") or {}).get("kind") == "moe"), None)
    E, top = (routed["router"]["experts"], routed["router"]["top"]) if routed else (1, 0)
    E_all = E + (routed["router"].get("identity", 0) if routed else 0)
    share = top * E / E_all                     # real experts a token uses (identities cost nothing)

    def step(news, before):
        """One step that brings `news` tokens to sequences that hold `before`."""
        T = sum(news)
        touched = E * (1.0 - (1.0 - share / E) ** T)
        size = (dense + head) * elem + expert / E * touched * elem + T * W * elem + len(news) * spec.vocab_size * 4
        flops = 2.0 * T * (dense + passes + expert / E * share) + 2.0 * len(news) * head
        for i in runs:
            m = layers[i]["mixer"]
            kind = layers[i]["type"]
            parts = [m["left"], m["right"]] if kind == "parallel" else [m]
            for p in parts:
                H, D, V = p.get("heads", 1), p.get("dim", 0), p.get("vdim", 0)
                if kind in ("delta", "channel_delta") or "tau" in p:
                    flops += T * H * D * V * (4 if "tau" in p else 6)
                    size += len(news) * H * D * V * 8
                elif kind == "mamba2":
                    flops += T * H * V * p["state"] * 5
                    size += len(news) * H * V * p["state"] * 8
                elif kind == "rglru":
                    flops += T * p["width"] * 4
                    size += len(news) * p["width"] * 8
                else:
                    maps = 2 if "diff" in p else 1
                    wide = D + p.get("rot_dim", 0)
                    seen = sum(visible_keys(p, b + j) for n, b in zip(news, before) for j in range(n))
                    flops += 2.0 * seen * H * maps * (wide + V)
                    row = p["kv_rank"] + p.get("rot_dim", 0) if "kv_rank" in p else p["kv_heads"] * (maps * D + V)
                    size += row * elem * (T + sum(min(visible_keys(p, b), b) for b in before))
        return size, flops

    prompts = lengths(c)
    if c["what"] == "decode":
        total = [step([1] * len(prompts), prompts)]
    else:
        total = [step(prompts, [0] * len(prompts))]
        total += [step([1] * len(prompts), [n + j for n in prompts]) for j in range(c["new"])]
    return {"bytes": float(sum(t[0] for t in total)), "flops": float(sum(t[1] for t in total))}


def tolerance(c):
    # about four times what these passes are off `exact`: float32 sums; bfloat16 rows between float32 sums
    return {"rel": 2e-5} if c["dtype"] == "float32" else {"rel": 3e-2}


# ---------------------------------------------------------------- the same in 64 bits
class Exact:
    """Plain formulas of the seven designs over one whole sequence, float64."""

    def __init__(self, c, seed):
        self.c, self.raw = c, config(c)
        self.width = self.raw.get("width", self.raw.get("hidden_size"))
        self.seed = seed
        self.eps = self.raw["norm"]["eps"] if "norm" in self.raw else self.raw["rms_norm_eps"]
        self.keep = {}

    def w(self, name, *shape):
        """A stored tensor in 64 bits; small ones are kept from sequence to sequence."""
        if name not in self.keep:
            t = weight(name, shape, self.c, self.seed, self.width)
            if t.numel() > 1 << 27:
                return t.double()
            self.keep[name] = t
        return self.keep[name].double()

    def rms(self, x, w=None):
        y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + self.eps)
        return y if w is None else y * w

    # ---- attention
    @staticmethod
    def attend(q, k, v, see, scale, cap=None, bias=None, sink=None):
        """q [T, H, D], k [T, G, D], v [T, G, V] -> [T, H, V]; bias [T, T, H]; sink [H]."""
        T, H, G = q.shape[0], q.shape[1], k.shape[1]
        out = torch.empty(T, H, v.shape[2], dtype=q.dtype, device=q.device)
        for h in range(H):
            s = (q[:, h] @ k[:, h // (H // G)].T.contiguous()) * scale
            if bias is not None:
                s = s + bias[:, :, h]
            if cap:
                s = cap * torch.tanh(s / cap)
            s = s.masked_fill(~see, -math.inf)
            top = s.amax(-1, keepdim=True)
            if sink is not None:
                top = torch.maximum(top, sink[h])
            s = torch.exp(s - top)
            total = s.sum(-1, keepdim=True)
            if sink is not None:
                total = total + torch.exp(sink[h] - top)
            out[:, h] = (s / total) @ v[:, h // (H // G)]
        return out

    @staticmethod
    def see(T, m, chunks):
        i = torch.arange(T, device="cuda")[:, None]
        j = torch.arange(T, device="cuda")[None, :]
        ok = j <= i
        mask = m.get("mask")
        if mask and chunks:
            ok = ok & (i // mask["size"] == j // mask["size"])
        elif mask:
            ok = ok & ((i - j < mask["size"]) | (j < mask.get("keep_first", 0)))
        return ok

    @staticmethod
    def turn(x, rot, halves=False, ramp=False):
        """Rotation of the first rot.dims entries of x [T, heads, D] at positions 0 .. T - 1."""
        dims, base, sc = rot["dims"], rot["base"], rot.get("scaling")
        f = [base ** (-2.0 * i / dims) for i in range(dims // 2)]
        grow = 1.0
        if sc and ramp:
            def pair(times):
                return dims * math.log(sc["original"] / (2.0 * math.pi * times)) / (2.0 * math.log(base))
            lo, hi = max(math.floor(pair(sc["fast"])), 0), min(math.ceil(pair(sc["slow"])), dims - 1)
            share = [min(1.0, max(0.0, (i - lo) / max(hi - lo, 0.001))) for i in range(dims // 2)]
            f = [a / sc["factor"] * s + a * (1.0 - s) for a, s in zip(f, share)]
            grow = 0.1 * math.log(sc["factor"]) + 1.0
        elif sc and "low" in sc:
            def slowed(a):
                wave = 2.0 * math.pi / a
                if wave < sc["original"] / sc["high"]:
                    return a
                if wave > sc["original"] / sc["low"]:
                    return a / sc["factor"]
                s = (sc["original"] / wave - sc["low"]) / (sc["high"] - sc["low"])
                return (1.0 - s) * a / sc["factor"] + s * a
            f = [slowed(a) for a in f]
        elif sc:
            f = [a / sc["factor"] for a in f]
        angle = torch.arange(x.shape[0], device="cuda", dtype=torch.float64)[:, None] * torch.tensor(f, device="cuda", dtype=torch.float64)
        cos, sin = torch.cos(angle)[:, None] * grow, torch.sin(angle)[:, None] * grow
        out = x.clone()
        at = (slice(0, dims // 2), slice(dims // 2, dims)) if halves else (slice(0, dims, 2), slice(1, dims, 2))
        a, b = x[..., at[0]], x[..., at[1]]
        out[..., at[0]] = a * cos - b * sin
        out[..., at[1]] = b * cos + a * sin
        return out

    # ---- what several designs share
    @staticmethod
    def taps(x, w, b=None):
        K = w.shape[1]
        padded = torch.cat([x.new_zeros(K - 1, x.shape[1]), x])
        y = sum(padded[j:j + x.shape[0]] * w[:, j] for j in range(K))
        return y if b is None else y + b

    @staticmethod
    def walk(q, k, v, decay, beta=None):
        """q, k, decay [T, H, D], v [T, H, V]: S <- decay S; u = beta (v - S^T k) or v; S <- S + k u^T; o = S^T q."""
        S = q.new_zeros(q.shape[1], q.shape[2], v.shape[2])
        out = torch.empty_like(v)
        for t in range(q.shape[0]):
            S = S * decay[t][:, :, None]
            u = v[t] if beta is None else beta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
            S = S + k[t][:, :, None] * u[:, None, :]
            out[t] = (S * q[t][:, :, None]).sum(1)
        return out

    def latent(self, h, p, m, halves, gate):
        """Keys and values from one latent a token; gate "head", "entry" or None."""
        T, W = h.shape
        H, D, V, rank, R = m["heads"], m["dim"], m["vdim"], m["kv_rank"], m.get("rot_dim", 0)
        if "q_rank" in m:
            n = m["q_rank"]
            q = self.rms(h @ self.w(p + "dq", n, W).T, self.w(p + "dq.norm", n)) @ self.w(p + "uq", H * (D + R), n).T
        else:
            q = h @ self.w(p + "q", H * (D + R), W).T
        q = q.view(T, H, D + R)
        down = h @ self.w(p + "dkv", rank + R, W).T
        lat = self.rms(down[:, :rank], self.w(p + "dkv.norm", rank))
        k = (lat @ self.w(p + "uk", H * D, rank).T).view(T, H, D)
        v = (lat @ self.w(p + "uv", H * V, rank).T).view(T, H, V)
        if R:
            k = torch.cat([k, self.turn(down[:, None, rank:], m["rot"], halves).expand(T, H, R)], -1)
            q = torch.cat([q[..., :D], self.turn(q[..., D:], m["rot"], halves)], -1)
        sink = self.w(p + "sink", H) if "q_rank" in m and R else None
        o = self.attend(q, k, v, self.see(T, m, False), m["scale"], sink=sink)
        if gate == "head":
            o = o * torch.sigmoid(h @ self.w(p + "g", H, W).T)[:, :, None]
        elif gate == "entry":
            o = o * torch.sigmoid(h @ self.w(p + "g", H * V, W).T).view(T, H, V)
        return o.reshape(T, H * V) @ self.w(p + "o", W, H * V).T

    def heads(self, h, p, m, biased=False, maps=1):
        T, W = h.shape
        H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        got = []
        for name, rows in (("q", H * maps * D), ("k", G * maps * D), ("v", G * V)):
            y = h @ self.w(p + name, rows, W).T
            got.append(y + self.w(p + name + ".b", rows) if biased else y)
        return got[0].view(T, H * maps, D), got[1].view(T, G * maps, D), got[2].view(T, G, V)

    def experts(self, h, p, mlp, score, unit):
        """score(h) -> (chosen [T, top], weights [T, top]); experts from E on are the identity."""
        E, ff, W = mlp["router"]["experts"], mlp["expert"]["ff"], h.shape[1]
        chosen, weights = score(h)
        out = torch.zeros_like(h)
        for e in range(E):
            row, place = (chosen == e).nonzero(as_tuple=True)
            if row.numel():
                q = f"{p}e{e}."
                y = unit(h[row], self.w(q + "gate", ff, W), self.w(q + "up", ff, W), self.w(q + "down", W, ff))
                out.index_add_(0, row, y * weights[row, place][:, None])
        same = torch.where(chosen >= E, weights, torch.zeros_like(weights)).sum(-1, keepdim=True)
        return out + same * h

    @staticmethod
    def grouped(scores, correction, r, worth):
        choice = scores + correction
        g = r["groups"]
        parts = choice.view(choice.shape[0], g["count"], -1)
        best = parts.topk(worth, -1).values.sum(-1).topk(g["keep"], -1).indices
        allowed = torch.zeros(parts.shape[:2], dtype=torch.bool, device=choice.device).scatter_(1, best, True)
        masked = parts.masked_fill(~allowed[:, :, None], -math.inf).view_as(choice)
        return masked.topk(r["top"], -1).indices

    @staticmethod
    def silu_unit(h, gate, up, down):
        return (torch.nn.functional.silu(h @ gate.T) * (h @ up.T)) @ down.T

    # ---- the designs: logits of a sequence at `rows`
    def forward(self, ids, rows):
        return getattr(self, self.c["family"])(torch.tensor(ids, device="cuda"), rows)

    def table(self, name, ids, vocab, width):
        return self.w(name, vocab, width)[ids]

    def qwen3(self, ids, rows):
        r = self.raw
        W, H, G, ff, V = r["hidden_size"], r["num_attention_heads"], r["num_key_value_heads"], r["intermediate_size"], r["vocab_size"]
        x = self.table("model.embed_tokens.weight", ids, V, W)
        T = x.shape[0]
        see = self.see(T, {}, False)
        rot = {"dims": 128, "base": r["rope_theta"]}
        for i in range(r["num_hidden_layers"]):
            p = f"model.layers.{i}."
            a = p + "self_attn."
            h = self.rms(x, self.w(p + "input_layernorm.weight", W))
            q, k, v = ((h @ self.w(a + n + "_proj.weight", g * 128, W).T).view(T, g, 128) for n, g in (("q", H), ("k", G), ("v", G)))
            q = self.turn(self.rms(q, self.w(a + "q_norm.weight", 128)), rot, True)
            k = self.turn(self.rms(k, self.w(a + "k_norm.weight", 128)), rot, True)
            o = self.attend(q, k, v, see, 128 ** -0.5)
            x = x + o.view(T, H * 128) @ self.w(a + "o_proj.weight", W, H * 128).T
            h = self.rms(x, self.w(p + "post_attention_layernorm.weight", W))
            m = p + "mlp."
            x = x + self.silu_unit(h, self.w(m + "gate_proj.weight", ff, W), self.w(m + "up_proj.weight", ff, W),
                                   self.w(m + "down_proj.weight", W, ff))
        x = self.rms(x[rows], self.w("model.norm.weight", W))
        return x @ self.w("model.embed_tokens.weight" if r["tie_word_embeddings"] else "lm_head.weight", V, W).T

    def delta(self, h, p, m, channel):
        T, W = h.shape
        H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        silu = torch.nn.functional.silu
        q, k, v = (silu(self.taps(h @ self.w(p + n, g * d, W).T, self.w(p + n + ".conv", g * d, 4))).view(T, g, d)
                   for n, g, d in (("q", G, D), ("k", G, D), ("v", H, V)))
        q, k = (y * torch.rsqrt((y * y).sum(-1, keepdim=True) + 1e-6) for y in (q, k))
        beta = torch.sigmoid(h @ self.w(p + "b", H, W).T)
        rate = torch.exp(self.w(p + "A_log", H))
        if channel:
            n = W // 16
            z = h @ self.w(p + "a1", n, W).T @ self.w(p + "a2", H * D, n).T + self.w(p + "dt_bias", H * D)
            decay = torch.exp(-rate[:, None] * torch.nn.functional.softplus(z).view(T, H, D))
            gate = torch.sigmoid(h @ self.w(p + "g1", n, W).T @ self.w(p + "g2", H * V, n).T)
        else:
            z = h @ self.w(p + "a", H, W).T + self.w(p + "dt_bias", H)
            decay = torch.exp(-rate * torch.nn.functional.softplus(z))[:, :, None]
            gate = silu(h @ self.w(p + "g", H * V, W).T)
        wide = functools.partial(torch.repeat_interleave, repeats=H // G, dim=1)
        o = self.walk(wide(q) * D ** -0.5, wide(k), v, decay, beta)
        o = self.rms(o, self.w(p + "norm", V)) * gate.view(T, H, V)
        return o.view(T, H * V) @ self.w(p + "o", W, H * V).T

    def vipalorn(self, ids, rows):
        r, W = self.raw, self.width

        def norm(x, name):
            return torch.nn.functional.layer_norm(x, (W,), self.w(name, W), None, self.eps)

        def unit(h, gate, up, down):
            g, u = torch.clamp(h @ gate.T, max=7.0), torch.clamp(h @ up.T, -7.0, 7.0)
            return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ down.T
        x = norm(self.table("embed", ids, VOCAB, W), "embed.norm")
        for i, layer in enumerate(r["layers"]):
            p, mlp = f"l{i}.", layer["mlp"]
            h = norm(x, p + "norm1")
            mixed = self.delta(h, p + "mix.", layer["mixer"], False) if layer["type"] == "delta" else \
                self.latent(h, p + "mix.", layer["mixer"], True, "head")
            E, top = mlp["router"]["experts"], mlp["router"]["top"]

            def score(y):
                best = (y @ self.w(p + "mlp.router", E, W).T + self.w(p + "mlp.router.b", E)).topk(top, -1)
                return best.indices, torch.softmax(best.values, -1)
            x = x + r["residual_mult"] * (mixed + self.experts(h, p + "mlp.", mlp, score, unit))
        return norm(x[rows], "final.norm") @ self.w("embed", VOCAB, W).T

    def modasun(self, ids, rows):
        r, W = self.raw, self.width
        x = self.table("embed", ids, VOCAB, W) * r["embedding"]["scale"]
        T = x.shape[0]
        for i, layer in enumerate(r["layers"]):
            p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
            if layer["type"] == "attention":
                q, k, v = self.heads(x, p + "mix.", m)
                steps = torch.div(torch.arange(T, device="cuda") + 1, m["q_temp"]["every"], rounding_mode="floor")
                temp = 1.0 + m["q_temp"]["coef"] * torch.log(steps.double() + 1.0)
                o = self.attend(self.rms(q) * temp[:, None, None], self.rms(k), v, self.see(T, m, False), m["scale"])
                mixed = o.reshape(T, -1) @ self.w(p + "mix.o", W, m["heads"] * m["vdim"]).T
            else:
                mixed = self.delta(x, p + "mix.", m, True)
            x = self.rms(r["postln_alpha"] * x + mixed, 1.0 + self.w(p + "norm1", W))
            E, ff, q = mlp["router"]["experts"], mlp["expert"]["ff"], p + "mlp."

            def score(y):
                s = torch.sigmoid(y @ self.w(q + "router", E, W).T)
                chosen = self.grouped(s, self.w(q + "correction", E), mlp["router"], 2)
                got = s.gather(1, chosen)
                return chosen, got / (got.sum(-1, keepdim=True) + 1e-20)
            y = self.experts(x, q, mlp, score, self.silu_unit)
            shared = self.silu_unit(x, self.w(q + "shared.gate", ff, W), self.w(q + "shared.up", ff, W), self.w(q + "shared.down", W, ff))
            y = y + torch.sigmoid(x @ self.w(q + "shared.sg", 1, W).T) * shared
            x = self.rms(r["postln_alpha"] * x + y, 1.0 + self.w(p + "norm2", W))
        return self.rms(x[rows], 1.0 + self.w("final.norm", W)) @ self.w("embed", VOCAB, W).T

    def mefatar(self, ids, rows):
        W = self.width
        gelu = functools.partial(torch.nn.functional.gelu, approximate="tanh")
        x = self.table("embed", ids, VOCAB, W)
        T = x.shape[0]

        def unit(h, p, m):
            n = W // m["blocks"]
            y = gelu(h @ self.w(p + "y", W, W).T + self.w(p + "y.b", W))
            u = self.taps(h @ self.w(p + "x", W, W).T + self.w(p + "x.b", W), self.w(p + "conv", W, 4), self.w(p + "conv.b", W))
            opened = []
            for name in ("ra", "ri"):
                mats, bias = self.w(p + name, m["blocks"], n, n), self.w(p + name + ".b", m["blocks"], n)
                opened.append(torch.sigmoid(torch.cat([u[:, b * n:(b + 1) * n] @ mats[b].T + bias[b] for b in range(m["blocks"])], -1)))
            a = torch.exp(-8.0 * opened[0] * torch.nn.functional.softplus(self.w(p + "lam", W)))
            put = torch.sqrt(1.0 - a * a) * opened[1] * u
            S, out = torch.zeros_like(u[0]), torch.empty_like(u)
            for t in range(T):
                S = a[t] * S + put[t]
                out[t] = S
            return (out * y) @ self.w(p + "o", W, W).T

        def left(h, p, m):
            H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
            q, k, v = (self.taps(y.reshape(T, -1), self.w(p + n + ".conv", y[0].numel(), 4))
                       for n, y in zip("qkv", self.heads(h, p, m)))
            q = self.turn(self.rms(q, self.w(p + "q.norm", H * D)).view(T, H, D), m["rot"])
            k = self.turn(self.rms(k, self.w(p + "k.norm", G * D)).view(T, G, D), m["rot"])
            o = self.attend(q, k, v.view(T, G, V), self.see(T, m, False), m["scale"], sink=self.w(p + "sink", H))
            return (o.reshape(T, H * V) * torch.sigmoid(h @ self.w(p + "g", H * V, W).T)) @ self.w(p + "o", W, H * V).T

        def right(h, p, m):
            H, D, V, n = m["heads"], m["dim"], m["vdim"], m["rank"]
            q, k, v = ((h @ self.w(p + a, H * d, W).T).view(T, H, d) for a, d in (("q", D), ("k", D), ("v", V)))
            z = h @ self.w(p + "a1", n, W).T @ self.w(p + "a2", H * D, n).T + self.w(p + "a2.b", H * D)
            o = self.walk(q * D ** -0.5, k, v, (torch.sigmoid(z) ** (1.0 / m["tau"])).view(T, H, D))
            o = self.rms(o, self.w(p + "norm", V)).reshape(T, H * V)
            return (o * torch.nn.functional.silu(h @ self.w(p + "g", H * V, W).T)) @ self.w(p + "o", W, H * V).T
        for i, layer in enumerate(self.raw["layers"]):
            p, m, ff = f"l{i}.", layer["mixer"], layer["mlp"]["ff"]
            h = self.rms(x, self.w(p + "norm1", W))
            if layer["type"] == "rglru":
                mixed = unit(h, p + "mix.", m)
            else:
                mixed = 0.5 * (self.rms(left(h, p + "mix.left.", m["left"]), self.w(p + "mix.left.out", W))
                               + self.rms(right(h, p + "mix.right.", m["right"]), self.w(p + "mix.right.out", W)))
            x = x + self.w(p + "ls1", W) * mixed
            h, q = self.rms(x, self.w(p + "norm2", W)), p + "mlp."
            y = (gelu(h @ self.w(q + "gate", ff, W).T) * (h @ self.w(q + "up", ff, W).T)) @ self.w(q + "down", W, ff).T
            x = x + self.w(p + "ls2", W) * y
        return self.rms(x[rows], self.w("final.norm", W)) @ self.w("embed", VOCAB, W).T

    def bozasun(self, ids, rows):
        W, side, eps = self.width, self.raw["token_side"]["dim"], self.eps
        layers = self.raw["layers"]
        x = self.table("embed", ids, VOCAB, W)
        extra = self.table("side.embed", ids, VOCAB, len(layers) * side)
        T = x.shape[0]

        def space(h, p, m):
            H, P, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
            inner = H * P
            z, u, dt = (h @ self.w(p + "in", 2 * inner + 2 * G * N + H, W).T).split([inner, inner + 2 * G * N, H], -1)
            u = torch.nn.functional.silu(self.taps(u, self.w(p + "conv", inner + 2 * G * N, 4), self.w(p + "conv.b", inner + 2 * G * N)))
            v = u[:, :inner].reshape(T, H, P)
            B, C = (y.reshape(T, G, N).repeat_interleave(H // G, 1) for y in u[:, inner:].split(G * N, -1))
            dt = torch.nn.functional.softplus(dt + self.w(p + "dt_bias", H))
            decay = torch.exp(-torch.exp(self.w(p + "A_log", H)) * dt)[:, :, None]
            y = self.walk(C, B, v * dt[:, :, None], decay) + self.w(p + "D", H)[:, None] * v
            y = (y.reshape(T, inner) * torch.nn.functional.silu(z)).view(T, m["norm_groups"], -1)
            y = (y * torch.rsqrt((y * y).mean(-1, keepdim=True) + eps)).reshape(T, inner) * self.w(p + "norm", inner)
            return y @ self.w(p + "o", W, inner).T

        def attention(h, p, m):
            q, k, v = self.heads(h, p, m, biased=True)
            q = self.turn(self.rms(q, self.w(p + "q.norm", m["dim"])), m["rot"])
            k = self.turn(self.rms(k, self.w(p + "k.norm", m["dim"])), m["rot"])
            o = self.attend(q, k, v, self.see(T, m, True), m["scale"], cap=m["softcap"]).reshape(T, -1)
            return o @ self.w(p + "o", W, o.shape[1]).T + self.w(p + "o.b", W)
        for i, layer in enumerate(layers):
            p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
            h = self.rms(x, self.w(p + "norm1", W))
            if layer["type"] == "mamba2":
                x = x + space(h, p + "mix.", m)
            elif layer["type"] == "attention":
                x = x + attention(h, p + "mix.", m)
            else:
                x = x + self.latent(h, p + "mix.", m, False, "entry")
            n = mlp["router"]["experts"] + mlp["router"]["identity"]

            def score(y):
                s = torch.softmax(y @ self.w(p + "mlp.router", n, W).T, -1)
                chosen = self.grouped(s, self.w(p + "mlp.correction", n), mlp["router"], 1)
                return chosen, s.gather(1, chosen)
            x = x + self.experts(self.rms(x, self.w(p + "norm2", W)), p + "mlp.", mlp, score, self.silu_unit)
            y = torch.nn.functional.gelu(x @ self.w(p + "side.gate", side, W).T, approximate="tanh") * extra[:, i * side:(i + 1) * side]
            x = x + self.rms(y @ self.w(p + "side.proj", W, side).T, self.w(p + "side.norm", W))
        return self.rms(x[rows], self.w("final.norm", W)) @ self.w("head", VOCAB, W).T

    def passes(self):
        loop, n = self.raw["loop"], len(self.raw["layers"])
        order = [(i, None) for i in range(loop["start"])]
        for t in range(loop["times"]):
            order += [(i, t if i == loop["start"] else None) for i in range(loop["start"], loop["stop"])]
        return order + [(i, None) for i in range(loop["stop"], n)]

    def mutedra(self, ids, rows):
        r, W = self.raw, self.width
        first = x = self.table("embed", ids, VOCAB, W) * r["embedding"]["scale"]
        T = x.shape[0]

        def norm(y, name):
            return torch.tanh(self.w(name + ".alpha") * y) * self.w(name, W) + self.w(name + ".b", W)

        def attention(h, p, m):
            q, k, v = self.heads(h, p, m)
            half, most = 16, m["bias_max"]
            row = [n if n < half else min(31, half + math.floor(math.log(n / half) / math.log(most / half) * half)) for n in range(T)]
            i = torch.arange(T, device="cuda")
            bias = self.w(p + "rel", 32, m["heads"])[torch.tensor(row, device="cuda")[(i[:, None] - i[None, :]).clamp(min=0)]]
            o = self.attend(q, k, v, self.see(T, m, False), m["scale"], bias=bias, sink=q.new_zeros(m["heads"]))
            return o.reshape(T, -1) @ self.w(p + "o", W, m["heads"] * m["vdim"]).T
        for i, start in self.passes():
            if start is not None:
                x = x + (first if start else 0.0) + self.w("loop.step", r["loop"]["times"], W)[start]
            layer, p = r["layers"][i], f"l{i}."
            h, m, ff, q = norm(x, p + "norm1"), layer["mixer"], layer["mlp"]["ff"], p + "mlp."
            y = attention(h, p + "mix.", m) if layer["type"] == "attention" else \
                self.latent(h, p + "mix.", m, False, "head" if "rot_dim" in m else None)
            x = x + norm(y, p + "norm1b")
            h = norm(x, p + "norm2")
            y = (torch.relu(h @ self.w(q + "gate", ff, W).T) * (h @ self.w(q + "up", ff, W).T)) @ self.w(q + "down", W, ff).T
            x = x + norm(y, p + "norm2b")
        z = norm(x[rows], "final.norm") @ self.w("head", VOCAB, W).T
        return r["logit_softcap"] * torch.tanh(z / r["logit_softcap"])

    def figalorn(self, ids, rows):
        r, W = self.raw, self.width
        first = x = self.table("embed", ids, VOCAB, W)
        T = x.shape[0]

        def maps(h, p, m):
            H, G, D = m["heads"], m["kv_heads"], m["dim"]
            q, k, v = self.heads(h, p, m, biased=True, maps=2)
            q, k = self.turn(q, m["rot"]).view(T, H, 2, D), self.turn(k, m["rot"]).view(T, G, 2, D)
            dot = [(self.w(p + "lq" + n, D) * self.w(p + "lk" + n, D)).sum() for n in "12"]
            lam = torch.exp(dot[0]) - torch.exp(dot[1]) + m["diff"]
            o = [self.attend(q[:, :, j], k[:, :, j], v, self.see(T, m, True), m["scale"]) for j in range(2)]
            o = (self.rms(o[0] - lam * o[1]) * (1.0 - m["diff"])).reshape(T, -1)
            return (o * torch.sigmoid(h @ self.w(p + "g", o.shape[1], W).T)) @ self.w(p + "o", W, o.shape[1]).T

        def window(h, p, m):
            H, G, D = m["heads"], m["kv_heads"], m["dim"]
            q = (h @ self.w(p + "q", H * D, W).T).view(T, H, D)
            v = (h @ self.w(p + "k", G * D, W).T).view(T, G, D)
            q = self.turn(self.rms(q, self.w(p + "q.norm", D)), m["rot"], True, True)
            k = self.turn(self.rms(v, self.w(p + "k.norm", D)), m["rot"], True, True)
            o = self.attend(q, k, v, self.see(T, m, False), m["scale"], cap=m["softcap"]).reshape(T, -1)
            return o @ self.w(p + "o", W, H * D).T
        for i, start in self.passes():
            if start is not None:
                x = torch.cat([x, first], -1) @ self.w("loop.in", W, 2 * W).T
            layer, p = r["layers"][i], f"l{i}."
            h, ff = self.rms(x, 1.0 + self.w(p + "norm1", W)), layer["mlp"]["ff"]
            x = x + (window if layer["type"] == "attention_2" else maps)(h, p + "mix.", layer["mixer"])
            h = self.rms(x, 1.0 + self.w(p + "norm2", W))
            x = x + torch.nn.functional.gelu(h @ self.w(p + "mlp.up", ff, W).T) @ self.w(p + "mlp.down", W, ff).T
        return self.rms(x[rows], 1.0 + self.w("final.norm", W)) @ self.w("head", VOCAB, W).T


def exact(c, seed):
    prompts, steps = tokens(c, seed)
    model = Exact(c, seed)
    found = []
    few = c["what"] == "decode" and sum(map(len, prompts)) > 4000       # then the first sequence alone
    for i, p in enumerate(prompts[:1] if few else prompts):
        ids = p + [s[i] for s in steps]
        rows = list(range(len(p) if c["what"] == "decode" else len(p) - 1, len(ids)))
        found.append(model.forward(ids, rows))
    logits = torch.stack(found, 1)                                       # [steps, sequences, vocabulary]
    if c["what"] == "decode":
        return {"first": logits[0, :1], "rest": None if few else logits[0, 1:]}
    return list(logits)
