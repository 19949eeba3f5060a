"""The tokenizer's fp32 tiles at the batches where the choice changes: 64x64
convolutions (40 sequences: 41.25 row tiles) and 128x128 searches (129: 64.5 row
tiles at the last level), the rows past the last full tile included. Each
level's codes of the first and last sequences by oracle replay, as in
test_vq_tokenizer_gpu.py."""
import numpy as np
import pytest

from .test_vq_tokenizer_gpu import _check_codes, _model, _torch, vo

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch", [40, 129])
def test_wmt14_batches(batch):
    torch = _torch()
    ocfg, enc, qw, dec, tok = _model(vo.WMT14, seed=batch)
    ids = np.random.default_rng(batch).integers(0, ocfg.in_vocab, size=(batch, 64))
    print(f"vq_tok WMT14 B={batch}", flush=True)
    a = tok.encode(ids, want_latent=True)
    pick = [0, batch - 1]
    _check_codes(ocfg, qw, a["latent"][pick].cpu().numpy().astype(np.float64),
                 a["codes"][pick].cpu().numpy(), a["zhat"][pick].cpu().numpy())
    assert torch.equal(tok.reconstruct(a["codes"]), a["zhat"])
