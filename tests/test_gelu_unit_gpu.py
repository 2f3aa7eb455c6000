"""The gated unit with the tanh form of gelu in the epilogue of the gate/up product (csrc/gemm_mfma.hip): few rows, K slices, every
large tile, steps of 32 k, against float64."""
import pytest
import torch

from herbert_rs_amd.kernels import mfma

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("M,I,K", [(1, 64, 64), (5, 512, 2048), (16, 96, 96), (17, 512, 1024), (48, 1024, 2048), (130, 80, 96), (300, 512, 256),
                                   (700, 1536, 192), (1777, 3072, 128), (600, 72 * 16, 64)])
@pytest.mark.parametrize("packed", [False, True])
def test_gelu_unit(M, I, K, packed):
    """float32 sums of K terms of bfloat16 operands (K 2^-24 of the terms' sizes, which the unit passes on at most 1.13 times the other
    factor), the exponential's and the reciprocal's last places (2^-21), rounded to bfloat16 (eight bits: half a last place is up to 2^-8)."""
    g = torch.Generator().manual_seed(M + I)
    a = torch.randn(M, K, generator=g).bfloat16()
    a[0] *= 30.0                                            # (gates far out on either side)
    gate, up = ((torch.randn(I, K, generator=g) * K ** -0.5).bfloat16() for _ in range(2))
    w = mfma.interleave_gate_up(gate.to(DEV), up.to(DEV))
    out = torch.full((M, I), 7.0, dtype=torch.bfloat16, device=DEV)
    mfma.gemm_swiglu(a.to(DEV), mfma.pack_weight(w) if packed else w, out, packed=packed, activation="gelu_tanh")
    z, u = a.double() @ gate.double().T, a.double() @ up.double().T
    want = torch.nn.functional.gelu(z, approximate="tanh") * u
    off_z, off_u = (K * 2.0 ** -24 * (a.double().abs() @ m.double().abs().T) for m in (gate, up))
    bound = (2.0 ** -8 + 2.0 ** -20) * want.abs() + 1.13 * off_z * u.abs() + z.abs() * off_u + 1e-30
    off = (out.cpu().double() - want).abs()
    # (gelu of a gate below -6: the product is below 1e-8 of the gate, and the exponential's argument has an error of its own size)
    assert bool((off <= bound + 1e-6 * (z.abs() + 1) * (z < -3) * u.abs()).all()), float((off - bound).max())


def test_a_gate_beyond_the_exponentials_range():
    a = torch.ones(20, 64, dtype=torch.bfloat16, device=DEV)
    gate = torch.zeros(64, 64)
    gate[0, 0], gate[1, 0], gate[2, 0] = 1e20, -1e20, -60.0
    up = torch.zeros(64, 64)
    up[:, 0] = 1.0
    out = torch.empty(20, 64, dtype=torch.bfloat16, device=DEV)
    mfma.gemm_swiglu(a, mfma.interleave_gate_up(gate.bfloat16().to(DEV), up.bfloat16().to(DEV)), out, activation="gelu_tanh")
    assert bool((out[:, 0] == gate[0, 0].bfloat16().to(DEV)).all()) and bool((out[:, 1:] == 0).all())
