"""RMSNorm's register kernel at its widths and on both sides of the row count
up to which it loads the weight up front: bit-identical to the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [576, 896, 2560])
@pytest.mark.parametrize("rows", [1, 7, 2048, 2049])
def test_rms_norm_register_widths(ncm, oracle, cuda, rows, width):
    import torch
    from ncmorph_amd import kernels

    rng = np.random.default_rng(rows + width)
    x = (rng.standard_normal((rows, width)) * 3).astype(np.float32)
    w = (rng.standard_normal(width) * 0.1 + 1).astype(np.float32)
    xd, wd = torch.from_numpy(x).to(cuda), torch.from_numpy(w).to(cuda)
    sample = sorted({0, rows // 2, rows - 1})
    for mode, bf16 in (("f32", False), ("bf16_f32", True)):
        y = kernels.rms_norm_rows(xd, wd, 1e-5, out_mode=mode).cpu().numpy()
        for r in sample:
            ref = oracle.rms_norm(x[r], w, 1e-5, bf16=bf16)
            assert np.array_equal(y[r].view(np.uint32), ref.view(np.uint32)), (mode, r)
    bits = kernels.rms_norm_rows(xd, wd, 1e-5, out_mode="bf16").cpu().view(torch.int16)
    assert np.array_equal(bits.numpy().view(np.uint16).astype(np.uint32) << 16,
                          y.view(np.uint32))
