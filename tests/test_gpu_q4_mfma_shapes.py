"""Prefill-sized affine-Q4 matmul: tiles of 32 and of 64 tokens, rows of fewer than eight scale groups, group counts around
the chunk and the eights of the bias pass, tiles with missing rows and tokens; scales too far apart for one fp16 operand
range; and a token's bits in calls of other sizes.

The bound is the one the entry point states, 2^-20 * sum_c (|q_c s| + 16 |s| + |b|) |x_c| + 1e-6."""
import numpy as np
import pytest

from golden import cases
from test_gpu_q4_mfma import magnitude_sums, reference

pytestmark = pytest.mark.gpu
synth = cases.synth


def tile_tokens(R, B):
    """32 where that many tiles of 32 tokens x 256 rows still have a compute unit each."""
    return 32 if -(-B // 32) * -(-R // 256) <= 256 else 64


def blocks(R, B):
    """Blocks of 64 and of 32 tokens per 256 rows."""
    halves, row_tiles = -(-B // 32), -(-R // 256)
    work, wide = halves * row_tiles, halves // 2
    if tile_tokens(R, B) == 32: wide = 0
    elif 512 < work <= 768 and work - 256 // row_tiles * row_tiles <= 512: wide = min(wide, 256 // row_tiles)
    return wide, halves - 2 * wide


def name_of(wide, narrow):
    """What a launch of so many blocks reports."""
    if wide and narrow: return f"q4_mfma_kernel, {wide} blocks of 64 tokens and {narrow} of 32"
    return f"q4_mfma_kernel, tiles of {64 if wide else 32} tokens"


def matmul(pkg, vals, scales, biases, R, C, xs):
    got = pkg.lib.q4_matmul(vals, scales, biases, R, C, xs)
    assert pkg.lib.load().salt_mi355_last_kernel().decode() == name_of(*blocks(R, xs.shape[0]))
    return got


def check(pkg, oracle, vals, scales, biases, R, C, xs):
    got = matmul(pkg, vals, scales, biases, R, C, xs)
    want = reference(oracle, vals, scales, biases, R, C, xs)
    assert np.isfinite(got).all()
    bound = 2.0 ** -20 * magnitude_sums(vals, scales, biases, R, C, xs)[1] + 1e-6
    ratio = np.abs(got.astype(np.float64) - want) / bound
    print("max err / bound", float(ratio.max()), flush=True)
    assert (ratio <= 1.0).all()


@pytest.mark.parametrize("R,C,B", [
    (65, 64, 33), (300, 448, 65),               # one and seven scale groups
    (257, 512, 70), (130, 576, 33),             # eight and nine groups
    (200, 4096, 100), (70, 1088, 64),           # sixty-four and seventeen
    (16640, 192, 130), (16448, 704, 129),       # 64-token tiles; a last tile of one token
    # waves without rows beside two and three rounds of group sums (49, 97 and 128 groups, 48 to a round)
    (65, 3136, 33), (65, 6208, 40), (300, 8192, 70), (16449, 3136, 70),
])
def test_tile_forms(pkg, oracle, R, C, B):
    print(f"mfma forms R={R} C={C} B={B}", flush=True)
    vals, scales, biases = synth.q4_tensor(R, C, R + C + B)
    check(pkg, oracle, vals, scales, biases, R, C, synth.activations(C, B, 23))


@pytest.mark.parametrize("R,C,B", [(130, 576, 33), (300, 448, 65), (16640, 192, 130), (16448, 704, 129),
                                   (65, 6208, 33), (130, 3136, 65)])
def test_without_biases(pkg, oracle, R, C, B):
    print(f"mfma no biases R={R} C={C} B={B}", flush=True)
    vals, scales, _ = synth.q4_tensor(R, C, R + C + B)
    check(pkg, oracle, vals, scales, None, R, C, synth.activations(C, B, 24))


def test_both_tile_forms_are_reached():
    """The sizes in this file on both sides of the rule, with and without missing tokens in the second half of a tile."""
    small, large = [(65, 33), (300, 65), (200, 100), (130, 33)], [(16640, 130), (16448, 129), (16640, 120)]
    assert all(tile_tokens(*s) == 32 for s in small) and all(tile_tokens(*s) == 64 for s in large)


@pytest.mark.parametrize("R,C,B", [(100, 640, 40), (300, 2112, 70), (16640, 192, 130), (16500, 640, 120)])
@pytest.mark.parametrize("with_biases", [True, False])
def test_scales_far_apart(pkg, oracle, R, C, B, with_biases):
    """Groups of a row up to 2^70 apart.  All but the first token see zeros where the scales are large, so that only the
    small ones decide their outputs."""
    print(f"mfma windows R={R} C={C} B={B}", flush=True)
    vals, _, _ = synth.q4_tensor(R, C, 5)
    rng = np.random.default_rng(R)
    far = np.arange(C // 64) % 3 == 1
    exponent = np.where(far, 40, rng.integers(-12, -4, (R, C // 64)))
    exponent[:, 2::3] = np.where(rng.random((R, len(range(2, C // 64, 3)))) < 0.5, -30, -6)
    s = np.ldexp(rng.uniform(1.0, 2.0, (R, C // 64)), exponent).astype(np.float32)
    scales = (s.view(np.uint32) >> 16).astype(np.uint16).reshape(-1)
    biases = ((-7.5 * synth.bf16_bits_to_f32(scales)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    xs = synth.activations(C, B, 29)
    xs[1:, np.repeat(far, 64)] = 0.0
    check(pkg, oracle, vals, scales, biases if with_biases else None, R, C, xs)


@pytest.mark.parametrize("R,C,B", [(300, 640, 40), (16640, 256, 130)])
@pytest.mark.parametrize("kind", ["scale inf", "scale nan", "bias inf", "x inf", "x nan", "x 1e37", "scale 2^100", "scale subnormal"])
def test_extreme_values_stay_in_their_row_or_token(pkg, oracle, R, C, B, kind):
    """What is not finite makes the outputs of its row or token not finite and leaves the bits of all others alone; what is
    finite and extreme keeps the bound."""
    print(f"mfma {kind} R={R} C={C} B={B}", flush=True)
    vals, scales, biases = synth.q4_tensor(R, C, 5)
    xs = synth.activations(C, B, 6)
    plain = matmul(pkg, vals, scales, biases, R, C, xs)
    s, b, x, row, token = scales.reshape(R, -1).copy(), biases.reshape(R, -1).copy(), xs.copy(), 3, 5
    if kind == "scale inf": s[row, 1] = 0x7F80
    if kind == "scale nan": s[row, 1] = 0x7FC0
    if kind == "bias inf": b[row, 2] = 0xFF80
    if kind == "x inf": x[token, 70] = np.inf
    if kind == "x nan": x[token, 70] = np.nan
    if kind == "x 1e37": x[token] *= np.float32(1e36)
    if kind == "scale 2^100": s[row] = 0x7180; b[row] = 0xF300       # 2^100 and -8 times that
    if kind == "scale subnormal": s[row] = 1; b[row] = 0
    got = matmul(pkg, vals, s.reshape(-1), b.reshape(-1), R, C, x)
    hit = np.zeros((B, R), bool)
    if kind.startswith("x"): hit[token] = True
    else: hit[:, row] = True
    assert np.array_equal(got.view(np.uint32)[~hit], plain.view(np.uint32)[~hit])
    if "inf" in kind or "nan" in kind:
        assert not np.isfinite(got[hit]).any()
        return
    tokens, rows = ([token], np.arange(R)) if kind.startswith("x") else (np.arange(B), [row])
    pick = np.ascontiguousarray(vals.reshape(R, -1)[rows]).reshape(-1), s[rows].reshape(-1), b[rows].reshape(-1)
    want = reference(oracle, *pick, len(rows), C, x[tokens])
    bound = 2.0 ** -20 * magnitude_sums(*pick, len(rows), C, x[tokens])[1] + 1e-6
    assert (np.abs(got[np.ix_(tokens, rows)].astype(np.float64) - want) <= bound).all()


def test_token_bits_do_not_depend_on_the_call(pkg):
    """A prompt in one call and in pieces, from one token per tile to more tiles than compute units; the same rows as a
    smaller matrix."""
    R, C, B = 8200, 1088, 520
    print(f"mfma pieces R={R} C={C} B={B}", flush=True)
    vals, scales, biases = synth.q4_tensor(R, C, 9)
    xs = synth.activations(C, B, 10)
    whole = pkg.lib.q4_matmul(vals, scales, biases, R, C, xs).view(np.uint32)
    for first, n in ((0, 1), (0, 33), (7, 64), (100, 130), (200, 260), (455, 65)):
        piece = pkg.lib.q4_matmul(vals, scales, biases, R, C, xs[first:first + n])
        assert np.array_equal(piece.view(np.uint32), whole[first:first + n]), (first, n)
    mixed = np.concatenate((xs[40:41], 1e3 * xs[:40], xs[41:80]))                   # other company, same number of tokens
    other = pkg.lib.q4_matmul(vals, scales, biases, R, C, mixed).view(np.uint32)
    assert np.array_equal(other[0], whole[40]) and np.array_equal(other[41:], whole[41:80])
    rows = 300
    part = pkg.lib.q4_matmul(vals[:rows * C // 8], scales[:rows * C // 64], biases[:rows * C // 64], rows, C, xs[:200])
    assert np.array_equal(part.view(np.uint32), whole[:200, :rows])
