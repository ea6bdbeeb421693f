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


def check(pkg, oracle, vals, scales, biases, R, C, xs):
    got = pkg.lib.q4_matmul(vals, scales, biases, R, C, xs)
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
])
def test_tile_forms(pkg, oracle, R, C, B):
    print(f"mfma forms R={R} C={C} B={B}", flush=True)
    vals, scales, biases = synth.q4_tensor(R, C, R + C + B)
    check(pkg, oracle, vals, scales, biases, R, C, synth.activations(C, B, 23))


@pytest.mark.parametrize("R,C,B", [(100, 640, 40), (300, 2112, 70)])
def test_scales_far_apart(pkg, oracle, R, C, B):
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
    check(pkg, oracle, vals, scales, biases, R, C, xs)


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
