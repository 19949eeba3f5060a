"""SiLU in the bf16 mode without expf and the IEEE division: every finite bf16
gate against the float64 quotient, and fp32 gates across the range."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bf16(x):
    import torch

    return torch.from_numpy(x.astype(np.float32)).to(torch.bfloat16).view(torch.int16).numpy()


def test_silu_of_every_bf16(ncm, cuda):
    """bf16(silu(g)) differs from the correctly rounded one only where the
    quotient lies within a few fp32 ulps of a rounding boundary: expected in
    65,280 values about 65280 x 2 x 4 ulps / 65536 = 8, and by one step."""
    import torch
    from ncmorph_amd import kernels

    bits = np.arange(65536, dtype=np.uint32) << 16
    g = bits.view(np.float32)
    g = g[np.isfinite(g) & ((bits & 0x7F800000) != 0)]
    # Up to 88 the reference's own exp(-g) is finite in fp32.
    g = g[g > -88.5]
    exact = g.astype(np.float64) / (1.0 + np.exp(-g.astype(np.float64)))
    keep = np.abs(exact) >= 2.0**-126
    gd = torch.from_numpy(g).to(cuda)
    got = kernels.silu_mul(gd, torch.ones_like(gd), out_mode="bf16").cpu().view(torch.int16)
    diff = np.abs(got.numpy().astype(np.int32) - _bf16(exact).astype(np.int32))[keep]
    assert diff.max() <= 1 and np.count_nonzero(diff) <= 16, np.count_nonzero(diff)


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
    # Half a bf16 step (2^-9 of the value's binade) and the fp32 ulps beside it.
    assert np.all(np.abs(run(v) - exact) <= np.abs(exact) * (2.0**-8 + 2.0**-20))
