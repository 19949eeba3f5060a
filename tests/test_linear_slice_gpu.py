"""Few-row linears (csrc/linear_slice.hip: small tiles, K split over the
wavefronts): every tile it chooses between, at M, N and K around its edges.

Bars: every output within the D53 bound |y - y_f64| <= (K + 2) 2^-24 sum|x w|
(+ |bias|) of float64 (packages/kernels/root.zig:96-142), and bit for bit: the
bf16 modes and the residual are the fp32 result rounded / added, the fused
SwiGLU and RoPE are the plain product followed by the unfused kernels, and a
row's outputs do not depend on the rows beside it."""
import numpy as np
import pytest

from ncmorph_amd import synth

pytestmark = pytest.mark.gpu

# M, K, N: one row; each row-block count up to 5 and one past; K below one
# 64-element tile, ragged, and not a multiple of the 8 wavefronts' tiles; odd
# N, N below a tile and N of four rounds (two column blocks with up to 48 rows).
SHAPES = [(1, 8, 1), (1, 2048, 2048), (16, 72, 64), (17, 576, 576), (33, 1096, 130),
          (48, 520, 49153), (49, 64, 49153), (64, 4864, 897), (65, 896, 1152), (81, 2048, 3071),
          (130, 1536, 2048), (203, 1000, 2048), (300, 512, 2048), (512, 328, 2048),
          (600, 136, 2047), (640, 24, 1000)]


def _dev(rng, shape, std, cuda):
    import torch

    bits = synth.bf16_bits((rng.standard_normal(shape) * std).astype(np.float32))
    return torch.from_numpy(bits.view(np.int16).copy()).to(cuda).view(torch.bfloat16)


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_slice_outputs(ncm, cuda, m, k, n):
    import torch
    from ncmorph_amd import kernels

    print(f"slice m={m} k={k} n={n}", flush=True)
    rng = np.random.default_rng(m + k + n)
    x, w, b = _dev(rng, (m, k), 1.0, cuda), _dev(rng, (n, k), 0.05, cuda), _dev(rng, (n,), 0.5,
                                                                              cuda)
    y = kernels.linear_bf16(x, w, bias=b)
    ref = x.double() @ w.double().t() + b.double()
    bound = (x.double().abs() @ w.double().abs().t() + b.double().abs()) * (k + 2) * 2.0**-24
    assert bool(((y.double() - ref).abs() <= bound).all())
    want = y.to(torch.bfloat16)
    assert torch.equal(kernels.linear_bf16(x, w, bias=b, out_mode="bf16_f32"), want.float())
    y16 = kernels.linear_bf16(x, w, bias=b, out_mode="bf16")
    assert torch.equal(y16, want.view(torch.int16))
    h = torch.from_numpy(rng.standard_normal((m, n)).astype(np.float32)).to(cuda)
    h = h.to(torch.bfloat16).float()
    res = kernels.linear_bf16_residual(x, w, h, bias=b, out_mode="bf16_f32")
    assert torch.equal(res, (h + want.float()).to(torch.bfloat16).float())
    # The last row among other rows.
    x2 = x.clone()
    x2[:m - 1] = x2[:m - 1].flip(0)
    assert torch.equal(kernels.linear_bf16(x2, w, bias=b)[m - 1], y[m - 1])


@pytest.mark.parametrize("m,k,inter", [(1, 64, 32), (17, 576, 1536), (33, 520, 24608),
                                       (64, 1096, 4864), (77, 256, 2048), (203, 264, 1024)])
@pytest.mark.parametrize("bias", [False, True])
def test_slice_fused_epilogues(ncm, oracle, cuda, m, k, inter, bias):
    import torch
    from ncmorph_amd import kernels

    print(f"slice fused m={m} k={k} inter={inter} bias={bias}", flush=True)
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
    if rot:
        kernels.rope_rotate(ref[:, :rot], rot // 64, 64, seq, cd, sd)
    got = kernels.linear_bf16_rope64(x, w, rot, seq, cd, sd, bias=b)
    assert torch.equal(got.view(torch.int16), ref.view(torch.int16))
