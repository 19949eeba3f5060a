"""RMSNorm's register kernel (multiples of 32 past 64 and up to 5120) at the edges
of its register counts, where a row ends inside them, and on both sides of the
row count up to which it loads the weight up front: bit-identical to the
oracle, and nothing written past the last row."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width", [64, 96, 128, 256, 288, 576, 608, 768, 896, 1056, 1536, 1792,
                                   2080, 2560, 3072, 3584, 4064, 4128, 5120])
@pytest.mark.parametrize("rows", [1, 7, 2048, 2049])
def test_rms_norm_register_widths(ncm, oracle, cuda, rows, width):
    import torch
    from ncmorph_amd import kernels

    rng = np.random.default_rng(rows + width)
    x = (rng.standard_normal((rows, width)) * 3).astype(np.float32)
    w = (rng.standard_normal(width) * 0.1 + 1).astype(np.float32)
    xd, wd = torch.from_numpy(x).to(cuda), torch.from_numpy(w).to(cuda)
    sample = range(rows) if rows < 8 else sorted({0, rows // 2, rows - 1})

    def run(mode, dtype):
        buf = torch.full((rows * width + 64,), -77.0, dtype=dtype, device=cuda)
        kernels.rms_norm_rows(xd, wd, 1e-5, out_mode=mode, out=buf[:rows * width].view(rows, width))
        assert bool((buf[rows * width:] == -77.0).all())
        return buf[:rows * width].view(rows, width).cpu()

    for mode, bf16 in (("f32", False), ("bf16_f32", True)):
        y = run(mode, torch.float32).numpy()
        for r in sample:
            ref = oracle.rms_norm(x[r], w, 1e-5, bf16=bf16)
            assert np.array_equal(y[r].view(np.uint32), ref.view(np.uint32)), (mode, r)
    bits = run("bf16", torch.bfloat16).view(torch.int16)
    assert np.array_equal(bits.numpy().view(np.uint16).astype(np.uint32) << 16,
                          y.view(np.uint32))


def test_rms_norm_register_special_rows(ncm, oracle, cuda):
    """Rows of zeros, subnormal values, infinities and NaN at a width that ends
    inside the registers."""
    import torch
    from ncmorph_amd import kernels

    width = 1056
    x = np.random.default_rng(4).standard_normal((6, width)).astype(np.float32)
    x[0] = 0
    x[1] *= np.float32(1e-39)
    x[2, 1055] = np.inf
    x[3, 1024] = np.nan
    x[4] *= np.float32(1e19)
    w = np.ones(width, np.float32)
    for mode, bf16 in (("f32", False), ("bf16_f32", True)):
        y = kernels.rms_norm_rows(torch.from_numpy(x).to(cuda), torch.from_numpy(w).to(cuda), 1e-5,
                                  out_mode=mode).cpu().numpy()
        for r in range(6):
            ref = oracle.rms_norm(x[r], w, 1e-5, bf16=bf16)
            same = (y[r].view(np.uint32) == ref.view(np.uint32)) | (np.isnan(y[r]) & np.isnan(ref))
            assert same.all(), (mode, r)
