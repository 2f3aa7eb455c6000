"""The native call of an entry point: every argument arrives, whatever its kind and place."""
import ctypes
import random

import pytest
import torch

from herbert_rs_amd.errors import BackendError
from herbert_rs_amd.kernels import lib, ops


@pytest.mark.parametrize("seed", range(12))
def test_arguments_arrive(seed):
    """Callbacks with random mixes of up to 40 words and 8 floats: six registers hold the first words, eight the floats, the stack the rest."""
    rng = random.Random(seed)
    words, floats = [(0, 0), (40, 8), (6, 8), (7, 1), (1, 0), (0, 3)][seed] if seed < 6 else (rng.randint(0, 40), rng.randint(0, 8))
    kinds = [rng.choice((ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t, ctypes.c_uint32)) for _ in range(words)] + [ctypes.c_float] * floats
    rng.shuffle(kinds)
    given, want = [], []
    for k in kinds:
        if k is ctypes.c_float:
            v = rng.choice((0.0, -1.5, 3, 2.0 ** 100, float("inf")))
            given.append(v), want.append(float(v))
        elif k is ctypes.c_void_p:
            v = rng.choice((None, 0, rng.getrandbits(47)))
            given.append(v), want.append(v or None)
        elif k is ctypes.c_int:
            v = rng.choice((True, rng.randint(-2 ** 31, 2 ** 31 - 1)))
            given.append(v), want.append(int(v))
        else:
            v = rng.getrandbits(64 if k is ctypes.c_size_t else 32)
            given.append(v), want.append(v)
    seen = []

    @ctypes.CFUNCTYPE(ctypes.c_int, *kinds)
    def function(*args):
        seen.extend(args)
        return 7 + seed
    entry = lib.host().entry(ctypes.cast(function, ctypes.c_void_p).value, "".join("f" if k is ctypes.c_float else "i" for k in kinds))
    assert lib.host().invoke(entry, *given) == 7 + seed
    assert seen == want


def test_what_is_no_argument_is_refused():
    host = lib.host()
    with pytest.raises(ValueError):
        host.entry(1, "i" * 41)
    with pytest.raises(ValueError):
        host.entry(1, "f" * 9)
    entry = host.entry(1, "if")                             # (never reached)
    for bad in ((), (1,), (1, 2.0, 3), (1.5, 2.0), ("a", 2.0), (1, "b"), (1, None)):
        with pytest.raises(TypeError):
            host.invoke(entry, *bad)
    with pytest.raises((TypeError, ValueError)):
        host.invoke(3, 1, 2.0)
    with pytest.raises(BackendError, match="empty problem"):
        lib.call("gemm_plain", "hb_gemm_plain", None, 0, None, 0, None, 0, 0, 1, 1, 1, 1, 1, 0, None)


def test_an_entry_point_is_known_only_once_it_can_be_called(monkeypatch):
    """Another thread that finds it there calls it at once: also the first one ever."""
    class Entries(dict):
        def __setitem__(self, key, entry):
            super().__setitem__(key, entry)
            with pytest.raises(BackendError, match="empty problem"):
                lib.call(*key, None, 0, None, 0, None, 0, 0, 1, 1, 1, 1, 1, 0, None)
            tried.append(key)
    tried = []
    monkeypatch.setattr(lib, "_entries", Entries())
    monkeypatch.setattr(lib, "_invoke", None)
    with pytest.raises(BackendError, match="empty problem"):
        lib.call("gemm_plain", "hb_gemm_plain", None, 0, None, 0, None, 0, 0, 1, 1, 1, 1, 1, 0, None)
    assert tried == [("gemm_plain", "hb_gemm_plain")]


def test_a_tensor_off_the_gpu_is_refused():
    assert not lib.host().fits(torch.zeros(3), None, None) and not lib.host().fits(None, None, None)
    for wrong in (torch.zeros(3), 5, None):
        with pytest.raises(BackendError, match="rows must be a tensor on the GPU"):
            ops._check(wrong, "rows")


class Stubborn(torch.Tensor):
    """Says that it lies on the GPU and raises whatever else it is asked."""
    @staticmethod
    def __new__(cls, policy):
        return torch.Tensor._make_wrapper_subclass(cls, (2, 3), dtype=torch.float32, device="cuda", dispatch_sizes_strides_policy=policy)

    @classmethod
    def __torch_dispatch__(cls, func, types, args=(), kwargs=None):
        raise RuntimeError("not to be asked")


@pytest.mark.parametrize("policy", ["strides", "sizes"])
def test_a_tensor_that_raises_is_refused_with_its_own_error(policy):
    t = Stubborn(policy)
    assert lib.host().fits(t, torch.float32, (2, 3)) is False
    with pytest.raises(RuntimeError, match="not to be asked"):
        ops._check(t, "rows", torch.float32, (2, 3))


@pytest.mark.gpu
def test_what_an_operand_must_be():
    t = torch.zeros(3, 4, 5, device="cuda")
    for shape in ((3, 4, 5), (None, 4, None), t.shape, [3, None, 5], None):
        ops._check(t, "t", torch.float32, shape)
        ops._check(t, "t", None, shape)
    ops._check(torch.zeros((), device="cuda"), "t", None, ())
    for shape in ((3, 4), (3, 4, 6), (None, None, 4), (3, 4, 5, 1), ()):
        with pytest.raises(BackendError, match="t must have shape"):
            ops._check(t, "t", torch.float32, shape)
    with pytest.raises(BackendError, match="t must be torch.bfloat16, got torch.float32"):
        ops._check(t, "t", torch.bfloat16, (3, 4, 5))
    for view in (t.transpose(0, 1), t[:, :, ::2]):
        with pytest.raises(BackendError, match="t must be contiguous"):
            ops._check(view, "t")
