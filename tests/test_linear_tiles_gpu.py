"""The bf16 linear's tiles (256x256, 128x256, 128x128, 64x128) at sizes that
choose each, with partial tiles in both directions.

Bars: every output within the D53 bound |y - y_f64| <= (K + 2) 2^-24 (sum|x w| +
|bias|) of float64 (packages/kernels/root.zig:96-142), and bit for bit: the
tiles give each other's sums, the bf16 modes and the residual are the fp32
result rounded / added, and the fused SwiGLU and RoPE are the plain product
followed by the unfused kernels."""
import numpy as np
import pytest

from ncmorph_amd import synth

pytestmark = pytest.mark.gpu


def _dev(rng, shape, std, cuda):
    import torch

    bits = synth.bf16_bits((rng.standard_normal(shape) * std).astype(np.float32))
    return torch.from_numpy(bits.view(np.int16).copy()).to(cuda).view(torch.bfloat16)


# 64x128 (one round, two row tiles and six), 128x256 (one row tile, three, two
# rounds), 128x128, 256x256, 256x128 (three row tiles, nine in three rounds). Five row
# tiles (one band) of 64x128 and 128x256, nine of 256x256; the last with the
# residual's own tile order (2^24 elements or more, a grid that is no multiple of 8).
@pytest.mark.parametrize("m,k,n", [(128, 136, 16383), (350, 72, 5000), (77, 520, 9999), (128, 64, 49153),
                                   (300, 328, 40001), (1100, 8, 14000), (1500, 72, 2049), (600, 72, 15900),
                                   (600, 520, 9000), (2047, 200, 8190), (2300, 72, 7400), (300, 72, 6143),
                                   (600, 72, 12800), (2300, 72, 12000)])
def test_tile_outputs(ncm, cuda, m, k, n):
    import torch
    from ncmorph_amd import kernels

    print(f"tile m={m} k={k} n={n}", flush=True)
    rng = np.random.default_rng(m + k + n)
    x, w, b = _dev(rng, (m, k), 1.0, cuda), _dev(rng, (n, k), 0.05, cuda), _dev(rng, (n,), 0.5,
                                                                              cuda)
    y = kernels.linear_bf16(x, w, bias=b)
    rows = torch.unique(torch.cat([torch.arange(0, m, 7), torch.arange(max(0, m - 70), m)]))
    rows = rows.to(cuda)
    xr = x[rows].double()
    ref = xr @ w.double().t() + b.double()
    bound = (xr.abs() @ w.double().abs().t() + b.double().abs()) * (k + 2) * 2.0**-24
    assert bool(((y[rows].double() - ref).abs() <= bound).all())
    # The same rows in batches that choose other tiles.
    for copies in (2, 5):
        more = kernels.linear_bf16(torch.cat([x] * copies), w, bias=b)
        assert torch.equal(more[-m:], y) and torch.equal(more[:m], y)
    want = y.to(torch.bfloat16)
    assert torch.equal(kernels.linear_bf16(x, w, bias=b, out_mode="bf16_f32"), want.float())
    y16 = kernels.linear_bf16(x, w, bias=b, out_mode="bf16")
    assert torch.equal(y16, want.view(torch.int16))
    h = torch.from_numpy(rng.standard_normal((m, n)).astype(np.float32)).to(cuda)
    h = h.to(torch.bfloat16).float()
    res = kernels.linear_bf16_residual(x, w, h, bias=b, out_mode="bf16_f32")
    assert torch.equal(res, (h + want.float()).to(torch.bfloat16).float())


@pytest.mark.parametrize("m,k,inter", [(128, 136, 8192 - 32), (350, 72, 2560), (128, 64, 24608),
                                       (300, 200, 20000), (1100, 72, 7008), (1500, 64, 1056),
                                       (300, 72, 3072), (600, 72, 4512)])
@pytest.mark.parametrize("bias", [False, True])
def test_tile_fused_epilogues(ncm, oracle, cuda, m, k, inter, bias):
    import torch
    from ncmorph_amd import kernels

    print(f"tile fused m={m} k={k} inter={inter} bias={bias}", flush=True)
    rng = np.random.default_rng(m + k + inter)
    x, w = _dev(rng, (m, k), 1.0, cuda), _dev(rng, (2 * inter, k), 0.05, cuda)
    b = _dev(rng, (2 * inter,), 0.5, cuda) if bias else None
    gu = kernels.linear_bf16(x, w, bias=b, out_mode="bf16_f32").reshape(m, -1, 2, 32)
    want = kernels.silu_mul(gu[:, :, 0].contiguous(), gu[:, :, 1].contiguous(), out_mode="bf16")
    got = kernels.linear_bf16_swiglu(x, w, bias=b)
    assert torch.equal(got.view(torch.int16).reshape(-1), want.view(torch.int16).reshape(-1))

    seq = max(1, m // 3)
    cos, sin = oracle.rope_tables(oracle.rope_llama3(64, 500000.0, 32.0, 1.0, 4.0, 8192), seq)
    cd, sd = torch.from_numpy(cos).to(cuda), torch.from_numpy(sin).to(cuda)
    rot = (2 * inter) // 128 * 64
    ref = kernels.linear_bf16(x, w, bias=b, out_mode="bf16").view(torch.bfloat16)
    kernels.rope_rotate(ref[:, :rot], rot // 64, 64, seq, cd, sd)
    got = kernels.linear_bf16_rope64(x, w, rot, seq, cd, sd, bias=b)
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16))


# fp32: the 64x64 tiles at ragged M, N and K, and 128x128 in six rounds.
@pytest.mark.parametrize("m,k,n", [(700, 100, 8190), (333, 36, 30003), (500, 576, 49100)])
def test_f32_tiles(ncm, cuda, m, k, n):
    import torch
    from ncmorph_amd import kernels

    print(f"f32 tile m={m} k={k} n={n}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(m + k + n)
    x = torch.randn(m, k, generator=g, device=cuda)
    w = torch.randn(n, k, generator=g, device=cuda)
    y = kernels.linear_f32(x, w)
    ref = x.double() @ w.double().t()
    bound = (x.double().abs() @ w.double().abs().t()) * (k + 1) * 2.0**-24
    assert bool(((y.double() - ref).abs() <= bound).all())
