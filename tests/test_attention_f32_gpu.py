"""The f32 decoder's attention around its chunks of 128 (64) staged keys and its
panel of 2048 scores: one traced layer against the oracle's f32 composition,
the context within 1e-4 of its largest magnitude (the projections' sums differ
in order, as in test_decoder_f32_gpu.py)."""
import numpy as np
import pytest

from .decoder_f64 import random_model
from .test_decoder_f32_gpu import _dev, _f32_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hd,t,window", [(64, 1, 0), (64, 128, 0), (64, 129, 3), (32, 2048, 0),
                                         (64, 2057, 0), (32, 2177, 2100), (32, 2177, 130),
                                         (128, 257, 0), (256, 65, 0), (256, 200, 64)])
def test_context(ncm, oracle, cuda, hd, t, window):
    from ncmorph_amd import decoder

    print(f"f32 attention hd={hd} t={t} window={window}", flush=True)
    rng = np.random.default_rng(hd + t + window)
    hidden, inter, vocab, hq, hkv = 64, 64, 40, 2, 1
    embed, layers, fnorm = random_model(rng, lambda a: np.asarray(a, np.float32), hidden, inter,
                                        vocab, hq, hkv, hd, 1)
    spec = decoder.DecoderSpec(hidden=hidden, intermediate=inter, vocab=vocab, q_heads=hq,
                               kv_heads=hkv, head_dim=hd, layers=1, window=window,
                               rope_theta=10000.0)
    cos, sin = oracle.rope_tables(oracle.rope_default_frequencies(hd, 10000.0), t)
    ids = rng.integers(0, vocab, (1, t))
    w = _f32_weights(decoder, cuda, embed, layers, fnorm)
    _, tr = decoder.forward_f32(spec, w, ids, _dev(cos, cuda), _dev(sin, cuda), trace=True)
    trace = {}
    oracle.decoder_forward(ids[0], embed, layers, fnorm, None, cos, sin, hq, hkv, hd, 1e-5,
                           window=window, bf16=False, trace=trace)
    got, want = tr["attention_context"].cpu().numpy(), trace["attention_context"]
    assert np.max(np.abs(got - want)) <= 1e-4 * np.max(np.abs(want))
