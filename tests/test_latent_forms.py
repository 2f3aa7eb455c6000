"""Which form of the latent attention the sequences of a step take (kernels/latent.py), without a GPU."""
import numpy as np
import torch

from herbert_rs_amd.engine import StepEntry
from herbert_rs_amd.engine import batch as batching
from herbert_rs_amd.kernels import latent

KV = type("KV", (), {"k": torch.empty(0, dtype=torch.bfloat16), "page_size": 64})


def packed(held, new):
    return batching.pack([StepEntry(i, [0] * n, []) for i, n in enumerate(new)], [h - n for h, n in zip(held, new)], torch.device("cpu"))


def test_a_sequence_takes_the_form_that_it_takes_alone(monkeypatch):
    """Random steps: every sequence is in a call or in the rest, once, as it is alone; calls stay within their scratch, and the lists
    name the tiles and rows that are theirs."""
    sizes = (16, 128, 128, 512, 64)
    rng = np.random.default_rng(5)
    alone = {}

    def of(held, new):
        forms = latent.forms(packed(held, new), KV, *sizes)
        names = lambda which, n: list(range(len(held))) if which is None else which[:n].tolist()
        calls = [(names(c[0], c[1]),) + c[2:] for c in forms.calls]
        return calls, [(names(*part[:2]),) + part[2:] for part in forms.rest]
    assert of([300], [1]) == ([], []) and of([900, 900], [2, 2]) == ([], []) and not of([2, 7], [2, 7])[1]
    for bound in (256 << 20, 4 << 20):
        monkeypatch.setattr(latent, "HEADS_BYTES", bound)
        alone.clear()
        for _ in range(60):
            n = int(rng.integers(1, 9))
            new = np.exp(rng.uniform(0, 6.5, n)).astype(int).tolist()
            held = [k + int(h) for k, h in zip(new, rng.choice([0, 0, 50, 700, 5000], n))]
            calls, rest = of(held, new)
            built = sorted(i for names, *_ in calls for i in names)
            left = [i for names, *_ in rest for i in names]
            if not calls:
                left = list(range(n))
            assert sorted(built + left) == list(range(n)), (held, new)
            for i in range(n):
                key = (held[i], new[i])
                if key not in alone:
                    alone[key] = bool(of([held[i]], [new[i]])[0])
                assert alone[key] == (i in built), (key, held, new)
            for names, tiles, longest in calls:
                assert tiles == sum(-(-held[i] // 64) for i in names) and longest == max(new[i] for i in names)
                here = sum(2 * -(-held[i] // 64) * 64 * (16 * 256 + 64) + 4 * new[i] * 16 * 64 for i in names)
                there = sum(new[i] * 16 * (4 * 576 + 2 * 640) for i in names)
                assert here <= max(there, bound)
            starts = np.concatenate([[0], np.cumsum(new)])
            for names, first, rows, longest, context, apart in rest:
                assert first == starts[names[0]] and first + rows == starts[names[-1] + 1]
                assert longest == max(new[i] for i in names) and context == max(held[i] for i in names)
                assert apart or names == list(range(names[0], names[-1] + 1))
            runs = sum(1 for i in left if i - 1 not in left) if calls else 0
            assert len(rest) == (runs if runs <= latent.RUNS else 1) and all(part[-1] == (runs > latent.RUNS) for part in rest)
    assert [part[0] for part in of([900, 100, 900, 100, 900], [1, 100, 1, 100, 1])[1]] == [[0], [2], [4]]
    assert of([900, 100] * 4, [1, 100] * 4)[1][0][0] == [0, 2, 4, 6]
