"""SiLU in the bf16 mode: every bf16 gate against the float64 quotient, in the
SiLU x up kernel and in the fused SwiGLU epilogues, and fp32 gates across the
range."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bf16(x):
    import torch

    return torch.from_numpy(x.astype(np.float32)).to(torch.bfloat16).view(torch.int16).numpy()


def test_silu_of_every_bf16(ncm, cuda):
    """bf16(silu(g)) is the correctly rounded one for every gate whose quotient
    is a normal number (an fp32 quotient with expf and the IEEE division is
    within 1.2 ulps, and no bf16 gate's lies so near a rounding boundary). Below
    -88.5 the reference's own exp(-g) overflows in fp32: -0."""
    import torch
    from ncmorph_amd import kernels

    bits = np.arange(65536, dtype=np.uint32) << 16
    g = bits.view(np.float32)
    g = g[np.isfinite(g) & ((bits & 0x7F800000) != 0)]
    with np.errstate(over="ignore"):
        exact = g.astype(np.float64) / (1.0 + np.exp(-g.astype(np.float64)))
    gd = torch.from_numpy(g).to(cuda)
    got = kernels.silu_mul(gd, torch.ones_like(gd), out_mode="bf16").cpu().view(torch.int16)
    got = got.numpy()
    keep = (g >= -88.5) & (np.abs(exact) >= 2.0**-126)
    # Rounded from float64 in one step: 8 bits of the value's binade.
    step = 2.0 ** (np.floor(np.log2(np.abs(exact[keep]))) - 7)
    want = _bf16(np.rint(exact[keep] / step) * step)
    assert np.array_equal(got[keep], want), g[keep][got[keep] != want]
    assert (got[g < -88.5].view(np.uint16) == 0x8000).all()


@pytest.mark.parametrize("m", [1, 80, 300])
def test_fused_silu_of_every_bf16(ncm, cuda, m):
    """The fused epilogues (few-row and tile kernels) take the reciprocal and a
    correction instead of the division: the bits of the SiLU x up kernel for
    every gate, infinities and NaN included. Row i of the gate weight holds gate
    i, x selects it and an up projection of 1."""
    import torch
    from ncmorph_amd import kernels

    g = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    w = torch.zeros(65536 // 32, 2, 32, 8, dtype=torch.bfloat16)
    w[:, 0, :, 0] = g.reshape(-1, 32)
    w[:, 1, :, 1] = 1
    x = torch.zeros(m, 8, dtype=torch.bfloat16)
    x[:, :2] = 1
    got = kernels.linear_bf16_swiglu(x.to(cuda), w.reshape(-1, 8).to(cuda)).cpu()
    got = got.view(torch.int16)
    gd = g.float().to(cuda)
    want = kernels.silu_mul(gd, torch.ones_like(gd), out_mode="bf16").cpu().view(torch.int16)
    normal = ~((g.float().abs() < 2.0**-126) & (g.float() != 0))  # the product flushes these
    normal &= g.view(torch.int16) != -32768  # a sum of -0 and +0
    assert torch.equal(got[:, normal], want[normal].expand(m, -1))


def test_silu_limits_and_fp32_gates(ncm, cuda):
    import torch
    from ncmorph_amd import kernels

    def run(v):
        v = np.asarray(v, np.float32)
        gd = torch.from_numpy(v).to(cuda)
        return kernels.silu_mul(gd, torch.ones_like(gd), out_mode="bf16_f32").cpu().numpy()

    big = float(torch.tensor(3e38).to(torch.bfloat16))
    assert run([np.inf, 3e38, 0.0]).tolist() == [np.inf, big, 0.0]
    assert np.isnan(run([-np.inf, np.nan])).all()  # -inf / inf
    assert (run([-95.0, -200.0, -3e38]) == 0.0).all() and np.signbit(run([-200.0])).all()
    v = np.random.default_rng(5).uniform(-80, 80, 100000).astype(np.float32)
    exact = v.astype(np.float64) / (1.0 + np.exp(-v.astype(np.float64)))
    # Half a bf16 step is at most 2^-8 of the value; the fp32 ulps come beside it.
    assert np.all(np.abs(run(v) - exact) <= np.abs(exact) * (2.0**-8 + 2.0**-20))
