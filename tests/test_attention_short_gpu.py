"""Causal attention where the route changes with the size: the short kernel
(csrc/attention.hip: up to 256 keys, scores in registers) around its tiles of
32 keys and its two sizes, the one-block-per-workgroup launch past it, and
windows, against the oracle's bf16 core with the bound of the attention tests:
|dev - oracle| <= 2^-7 |ref| + 2^-7 max|v|, at least 99% equal bit for bit."""
import numpy as np
import pytest

from ncmorph_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,t,window", [(64, 1, 0), (64, 31, 0), (64, 33, 5), (64, 128, 0),
                                         (64, 129, 64), (64, 256, 33), (64, 257, 0),
                                         (128, 32, 0), (128, 97, 40), (128, 160, 0),
                                         (128, 255, 1), (128, 260, 0)])
def test_short_causal_attention(ncm, oracle, cuda, hd, t, window):
    import torch
    from ncmorph_amd import kernels

    print(f"short attention hd={hd} t={t} window={window}", flush=True)
    rng = np.random.default_rng(hd + t + window)
    batch, hq, hkv = 2, 4, 2
    bits = [synth.bf16_bits(rng.standard_normal((batch * t, n * hd)).astype(np.float32))
            for n in (hq, hkv, hkv)]
    q, k, v = (torch.from_numpy(b.view(np.int16)).to(cuda).view(torch.bfloat16) for b in bits)
    out = kernels.attention_bf16(q, k, v, batch, t, hq, hkv, hd, window=window).cpu().numpy()
    out16 = kernels.attention_bf16(q, k, v, batch, t, hq, hkv, hd, window=window,
                                   out_mode="bf16").cpu().view(torch.int16).numpy()
    assert np.array_equal(out16.view(np.uint16).astype(np.uint32) << 16, out.view(np.uint32))
    qf, kf, vf = (synth.bf16_to_f32(b) for b in bits)
    i = np.arange(t)
    mask = i[None, :] <= i[:, None]
    if window:
        mask &= i[None, :] > i[:, None] - window
    for b in range(batch):
        rows = slice(b * t, (b + 1) * t)
        ref = oracle.attention_core(qf[rows], kf[rows], vf[rows], mask, hq, hkv, hd, bf16=True)
        err = np.abs(out[rows] - ref)
        assert np.all(err <= 2.0**-7 * np.abs(ref) + 2.0**-7 * np.max(np.abs(vf[rows]))), b
        assert np.mean(out[rows] == ref) >= 0.99, np.mean(out[rows] == ref)


@pytest.mark.parametrize("hd,t", [(64, 77), (64, 256), (128, 130)])
def test_short_output_over_v(ncm, cuda, hd, t):
    """`out` may be v itself: every element of v is read before it is
    overwritten. Within the two kernels' difference (one rounding of a
    probability at 2^-8) of the same call with an output of its own."""
    import torch
    from ncmorph_amd import kernels

    g = torch.Generator(device=cuda).manual_seed(hd + t)
    batch, heads = 3, 4
    q, k, v = (torch.randn(batch * t, heads * hd, generator=g, device=cuda).to(torch.bfloat16)
               for _ in range(3))
    want = kernels.attention_bf16(q, k, v, batch, t, heads, heads, hd, out_mode="bf16")
    want, peak = want.float(), float(v.float().abs().max())
    for _ in range(3):
        w = v.clone()
        got = kernels.attention_bf16(q, k, w, batch, t, heads, heads, hd, out_mode="bf16", out=w)
        assert float((got.float() - want).abs().max()) <= 2.0**-7 * peak
    # Beside v in one buffer of rows.
    qkv = torch.cat([q, k, v], 1)
    cols = [slice(i * heads * hd, (i + 1) * heads * hd) for i in range(3)]
    got = kernels.attention_bf16(qkv[:, cols[0]], qkv[:, cols[1]], qkv[:, cols[2]], batch, t, heads,
                                 heads, hd, out_mode="bf16", out=qkv[:, cols[2]])
    assert float((got.float() - want).abs().max()) <= 2.0**-7 * peak
