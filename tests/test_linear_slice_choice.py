"""The few-row linears' choice of a tile (csrc/linear_slice.hip, linear_slice.h)
restated on the host: the shape lists of test_linear_slice_gpu.py reach every
tile that the choice can return, plain, in pairs (SwiGLU, RoPE) and in fp32."""
from .test_linear_slice_gpu import DECODER_F32, F32, FUSED, SHAPES

# Blocks of 16 rows and of 16 columns.
TILES = [(1, 1), (2, 1), (1, 2), (2, 2), (3, 2), (1, 4), (4, 2), (2, 4), (3, 4), (4, 4), (5, 4)]


def _cd(a, b):
    return -(-a // b)


def _tiles(t, m, n):
    return _cd(m, 16 * t[0]) * _cd(n, 16 * t[1])


def choose_bf16(m, n, paired=False):
    """(cost, tile): rounds of 256 CUs times the operand blocks loaded."""
    cost, tile = min(((_cd(_tiles(t, m, n), 256) * sum(t), i) for i, t in enumerate(TILES)
                      if t[1] > 1 or not paired))
    if m <= 48 and _cd(n, 64) > 768:
        tile = TILES.index((_cd(m, 16), 2))
    return cost, TILES[tile]


def fits_bf16(m, n, k):
    if m <= 64:
        return True
    cost, tile = choose_bf16(m, n)
    if tile == (5, 4) and (k <= 640 or (k <= 1024 and m <= 80)):
        return False
    return cost <= 13


def choose_f32(m, n, k, paired=False):
    """(estimated us, tile)."""
    def us(t):
        blocks, rounds = t[0] * t[1], _cd(_tiles(t, m, n), 256)
        one = 0.22 * blocks * 0.5 * ((_cd(k, 32) + 3) // 4) + 1.3 + 0.3 * blocks
        return 3.0 + (1.12 * rounds if rounds > 1 else 1.0) * one

    best, tile = min((us(t), i) for i, t in enumerate(TILES) if t[1] > 1 or not paired)
    return best, TILES[tile]


def fits_f32(m, n, k):
    rounds = _cd(_cd(m, 128) * _cd(n, 128), 256)
    large = rounds * (1.95 * _cd(k, 32) + 6.0)
    large = 3.0 + (0.9 * large if rounds >= 4 else large)
    small = 6.5 + _cd(_cd(m, 64) * _cd(n, 64), 256) * (0.5 * _cd(k, 32) + 0.6)
    us, _ = choose_f32(m, n, k)
    return us < large and us < 1.1 * small


def test_plain_bf16_tiles_are_all_reached():
    got = {choose_bf16(m, n)[1] for m, k, n in SHAPES if fits_bf16(m, n, k)}
    assert got == set(TILES), set(TILES) - got


def test_paired_bf16_tiles_are_all_reached():
    got = {choose_bf16(m, 2 * i, True)[1] for m, k, i in FUSED if fits_bf16(m, 2 * i, k)}
    assert got == {t for t in TILES if t[1] > 1}, got


def test_plain_f32_tiles_are_all_reached():
    got = {choose_f32(m, n, k)[1] for m, k, n in F32 if fits_f32(m, n, k)}
    assert got == set(TILES), set(TILES) - got


def test_f32_decoder_tiles_are_all_reached():
    pairs = {t for t in TILES if t[1] > 1}
    rope, swiglu = set(), set()
    for hidden, inter, hq, hkv, hd, t, _ in DECODER_F32:
        qkv, rows = (hq + 2 * hkv) * hd, 2 * t
        if hd == 64 and fits_f32(rows, qkv, hidden):
            rope.add(choose_f32(rows, qkv, hidden, True)[1])
        if fits_f32(rows, inter, hidden):
            swiglu.add(choose_f32(rows, 2 * inter, hidden, True)[1])
    assert rope == pairs, pairs - rope
    assert swiglu == pairs, pairs - swiglu
