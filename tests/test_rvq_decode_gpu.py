"""RVQ decode where its workgroups change shape: one row a thread and four (t a
multiple of 4, 2^26 elements or more), widths whose pieces fill the wavefronts
or leave lanes over, in one share or several, strides of 1, 2, 4 and more, and
level counts that leave every remainder of eight: bit-identical to the oracle."""
import numpy as np
import pytest

from ncmorph_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,t,d,strides,v", [
    (1, 4096, 64, (4, 2, 1), 40),
    (2, 2048, 576, (8, 4, 4, 2, 1), 300),
    (4, 1024, 320, (2, 1, 1), 17),
    (4, 1024, 512, (16, 8, 8, 4, 4, 2, 2, 1, 1), 33),
    (3, 1366, 128, (2, 1), 20),
    (1, 8, 2048, (8, 1), 5),
    (1, 33, 192, (1,) * 7, 9),
    (1, 37, 4160, (1,) * 3, 9),
    (2, 40, 1088, (8, 4, 4, 4, 4, 4), 9),
    # 2^26 elements and more: four rows a thread; the third one row (t odd).
    (4, 4100, 4096, (4, 2, 1), 12),
    (2, 16392, 2112, (8, 8, 4, 2, 2, 2, 1, 1, 1), 12),
    (1, 16387, 4096, (1, 1), 12),
])
def test_decode_shapes(ncm, oracle, cuda, b, t, d, strides, v):
    import torch
    from ncmorph_amd import vq

    print(f"rvq decode b={b} t={t} d={d} strides={strides}", flush=True)
    rng = np.random.default_rng(t + d)
    cb = synth.bf16_bits(rng.standard_normal((len(strides), v, d)).astype(np.float32))
    # Codes out of range are clamped.
    codes = rng.integers(-1, v + 1, (b, sum(t // s for s in strides))).astype(np.int32)
    got = vq.decode(torch.from_numpy(codes).to(cuda),
                    torch.from_numpy(cb.view(np.int16)).to(cuda).view(torch.bfloat16), strides, t)
    want = oracle.rvq_decode(np.clip(codes, 0, v - 1), cb, strides, t)
    assert np.array_equal(got.cpu().numpy().view(np.uint32), want.view(np.uint32))


def test_decode_of_many_narrow_rows(ncm, cuda):
    """More than 2^26 rows of 64 columns: the grid has 8 threads a row, of at
    most 2^32."""
    import torch
    from ncmorph_amd import vq

    t = 2**26 + 2
    cb = torch.arange(3 * 64, dtype=torch.float32, device=cuda).reshape(1, 3, 64)
    cb = cb.to(torch.bfloat16)
    codes = (torch.arange(t, dtype=torch.int32, device=cuda) * 7 % 3).reshape(1, t)
    got = vq.decode(codes, cb, (1,), t)
    for r0 in range(0, t, 2**24):
        want = cb[0].float()[codes[0, r0:r0 + 2**24].long()]
        assert torch.equal(got[0, r0:r0 + 2**24], want), r0


@pytest.mark.parametrize("b,t,d,levels,v", [(1, 1, 64, 1, 1), (1, 128, 256, 4, 512),
                                            (2, 33, 320, 3, 65), (1, 40, 512, 2, 511),
                                            (2, 128, 128, 3, 1024), (1, 257, 64, 2, 65),
                                            (2, 10, 448, 3, 500), (1, 9, 576, 2, 64)])
def test_full_resolution_encode(ncm, oracle, cuda, b, t, d, levels, v):
    """Encodes whose levels are all at full resolution run in one launch while
    they are small: codes and reconstruction bit-identical to the oracle, with
    the lowest index for duplicate codewords, and forced codes followed."""
    import torch
    from ncmorph_amd import vq

    print(f"rvq full resolution b={b} t={t} d={d} levels={levels} v={v}", flush=True)
    x, cb = synth.rvq_inputs(b * t + d, b, t, d, levels, v)
    cb[:, v // 2] = cb[:, 0]
    strides = (1,) * levels
    xd = torch.from_numpy(x).to(cuda)
    cbd = torch.from_numpy(cb.view(np.int16)).to(cuda).view(torch.bfloat16)
    ref = oracle.rvq_encode(x, cb, strides)
    r = vq.encode(xd, cbd, strides, want_gap=False)
    assert np.array_equal(r["codes"].cpu().numpy(), ref["codes"])
    assert np.array_equal(r["recon"].cpu().numpy().view(np.uint32), ref["recon"].view(np.uint32))
    force = np.random.default_rng(d).integers(0, v, (b, levels * t)).astype(np.int32)
    forced = oracle.rvq_encode(x, cb, strides, forced=force)
    r = vq.encode(xd, cbd, strides, want_gap=False, force_codes=torch.from_numpy(force).to(cuda))
    assert np.array_equal(r["codes"].cpu().numpy(), forced["codes"])
    assert np.array_equal(r["recon"].cpu().numpy().view(np.uint32),
                          forced["recon"].view(np.uint32))


@pytest.mark.parametrize("want_gap", [False, True])
def test_forced_codes_in_the_output(ncm, cuda, want_gap):
    """force_codes may be the codes output: every code is the library's own by
    the time it is read, so the encode is the unforced one, in the one launch
    of few rows as in the general path."""
    import torch
    from ncmorph_amd import vq

    x, cb = synth.rvq_inputs(3, 1, 100, 192, 4, 500)
    xd = torch.from_numpy(x).to(cuda)
    cbd = torch.from_numpy(cb.view(np.int16)).to(cuda).view(torch.bfloat16)
    own = vq.encode(xd, cbd, (1,) * 4, want_gap=want_gap)
    for _ in range(3):
        buf = torch.zeros((1, 400), dtype=torch.int32, device=cuda)
        r = vq.encode(xd, cbd, (1,) * 4, want_gap=want_gap, force_codes=buf, out={"codes": buf})
        assert torch.equal(r["codes"], own["codes"]) and torch.equal(r["recon"], own["recon"])


@pytest.mark.parametrize("d,v", [(64, 65), (320, 300)])
def test_full_resolution_rows_without_a_distance(ncm, oracle, cuda, d, v):
    """Rows that hold NaN or infinities get the codes of the general path,
    which an encode that asks for its gaps takes; a row whose squares overflow
    gets the oracle's."""
    import torch
    from ncmorph_amd import vq

    print(f"rvq rows without a distance d={d} v={v}", flush=True)
    x, cb = synth.rvq_inputs(d, 1, 8, d, 2, v)
    x[0, 1, 3] = np.nan
    x[0, 2, 5] = np.inf
    x[0, 3, d - 1] = -np.inf
    x[0, 5] = 0
    cbd = torch.from_numpy(cb.view(np.int16)).to(cuda).view(torch.bfloat16)
    got = vq.encode(torch.from_numpy(x).to(cuda), cbd, (1, 1), want_gap=False)
    want = vq.encode(torch.from_numpy(x).to(cuda), cbd, (1, 1), want_gap=True)
    assert np.array_equal(got["codes"].cpu().numpy(), want["codes"].cpu().numpy())
    assert np.array_equal(got["recon"].cpu().numpy(), want["recon"].cpu().numpy())

    x[0, 1:4] = x[0, 4] * 1e25
    ref = oracle.rvq_encode(x, cb, (1, 1))
    got = vq.encode(torch.from_numpy(x).to(cuda), cbd, (1, 1), want_gap=False)
    assert np.array_equal(got["codes"].cpu().numpy(), ref["codes"])
