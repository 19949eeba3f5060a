"""Few-row linears (csrc/linear_slice.hip: small tiles, K split over the
wavefronts): every tile it chooses between, at M, N and K around its edges
(test_linear_slice_choice.py holds these lists to that).

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
          (600, 136, 2047), (640, 24, 1000),
          # 2 x 1, 1 x 2, 1 x 4, 2 x 2, 3 x 2, 4 x 2, 2 x 4, 3 x 4 and 5 x 4 blocks.
          (20, 72, 2063), (3, 1000, 4113), (5, 264, 8209), (19, 72, 4113), (40, 136, 4113),
          (50, 72, 4099), (65, 136, 4113), (70, 72, 5457), (130, 648, 5457)]
FUSED = [(1, 64, 32), (17, 576, 1536), (33, 520, 24608), (64, 1096, 4864), (77, 256, 2048),
         (203, 264, 1024),
         # 2 x 2, 1 x 4, 2 x 4, 3 x 4 and 5 x 4 blocks, the last also at a model's size.
         (20, 72, 2080), (5, 72, 4128), (19, 136, 4128), (35, 72, 4128), (130, 648, 2752), (77, 1096, 8192)]
# K below, at and past one round of the wavefronts' 32-element tiles; N of one
# and of several rounds; the last of the first line past the small tiles' range.
F32 = [(1, 4, 1), (17, 576, 960), (33, 260, 1153), (77, 4864, 896), (200, 576, 577),
       (300, 1000, 4864), (600, 36, 130), (130, 896, 20000),
       (20, 36, 2113), (1, 36, 4161), (19, 36, 4161), (34, 36, 5505), (34, 36, 4161),
       (50, 36, 4161), (67, 36, 4161), (67, 132, 5505), (100, 1000, 5505), (131, 260, 5505)]
# hidden, intermediate, q heads, kv heads, head_dim, tokens of each of two
# sequences, biases.
DECODER_F32 = [(128, 256, 4, 2, 64, 37, True), (576, 1536, 9, 3, 64, 77, False),
               (96, 68, 3, 1, 32, 20, True), (576, 1536, 9, 3, 64, 100, True),
               (36, 4160, 63, 1, 64, 5, False), (36, 2112, 63, 1, 64, 10, True),
               (36, 4160, 63, 1, 64, 10, True), (36, 4160, 63, 1, 64, 17, False),
               (36, 2112, 63, 1, 64, 25, True), (36, 4160, 63, 1, 64, 25, False),
               (36, 4160, 63, 1, 64, 34, True), (36, 2752, 84, 1, 64, 17, True),
               (132, 4160, 84, 1, 64, 34, False), (260, 4160, 84, 1, 64, 65, True),
               (1000, 4160, 84, 1, 64, 50, False)]


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


@pytest.mark.parametrize("m,k,inter", FUSED)
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


@pytest.mark.parametrize("m,k,n", F32)
def test_slice_f32(ncm, cuda, m, k, n):
    import torch
    from ncmorph_amd import kernels

    print(f"slice f32 m={m} k={k} n={n}", flush=True)
    rng = np.random.default_rng(m + k + n)
    x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(cuda)
    w = torch.from_numpy(rng.standard_normal((n, k)).astype(np.float32)).to(cuda)
    y = kernels.linear_f32(x, w)
    ref = x.double() @ w.double().t()
    bound = (x.double().abs() @ w.double().abs().t()) * (k + 1) * 2.0**-24
    assert bool(((y.double() - ref).abs() <= bound).all())


@pytest.mark.parametrize("hidden,inter,hq,hkv,hd,t,biases", DECODER_F32)
def test_f32_decoder_fused_equals_traced(ncm, oracle, cuda, hidden, inter, hq, hkv, hd, t,
                                         biases):
    """Without a trace the f32 layers run one q|k|v product with the rotation,
    gate|up with the activation and the residual adds inside the products; with
    every stage traced those run apart. The same bits."""
    import torch
    from ncmorph_amd import decoder

    print(f"f32 decoder fused hidden={hidden} hd={hd} t={t}", flush=True)
    g = torch.Generator(device=cuda).manual_seed(hidden + t)

    def r(*shape, std=0.1):
        return torch.randn(*shape, generator=g, device=cuda) * std

    qkv = (hq + 2 * hkv) * hd
    layers = []
    for _ in range(2):
        layer = {"input_norm": 1 + r(hidden), "qkv_weight": r(qkv, hidden),
                 "o_weight": r(hidden, hq * hd), "post_attention_norm": 1 + r(hidden),
                 "gate_weight": r(inter, hidden), "up_weight": r(inter, hidden),
                 "down_weight": r(hidden, inter)}
        if biases:
            layer.update(qkv_bias=r(qkv), o_bias=r(hidden), gate_bias=r(inter),
                         up_bias=r(inter), down_bias=r(hidden))
        layers.append(layer)
    spec = decoder.DecoderSpec(hidden=hidden, intermediate=inter, vocab=200, q_heads=hq,
                               kv_heads=hkv, head_dim=hd, layers=2, rope_theta=10000.0)
    w = decoder.DecoderWeights(embed=r(200, hidden), final_norm=1 + r(hidden), layers=layers,
                               mode="f32")
    cos, sin = oracle.rope_tables(oracle.rope_default_frequencies(hd, 10000.0), t)
    tables = torch.from_numpy(cos).to(cuda), torch.from_numpy(sin).to(cuda)
    ids = np.random.default_rng(t).integers(0, 200, (2, t))
    plain = decoder.forward_f32(spec, w, ids, *tables)
    traced, _ = decoder.forward_f32(spec, w, ids, *tables, trace=True)
    assert torch.equal(plain, traced)
