"""The ordered sum of squares adds most parts of a vector by what they would add to a guess of the chain's value.  Replayed here
in fp32 with the parts and the scan of the kernel: the vectors that its GPU test calls stagnant and overtaking do make a guess
that lies on the other side of a power of two, after which every part has to be walked, and ordinary ones do not."""
import numpy as np
import pytest

from golden import cases
from test_gpu_ordered_sum import vector

f32 = np.float32


def scan(v):
    """Inclusive sums over 64 lanes: rows of 16 by shifts of 1, 2, 4, 8, then lane 15 of rows 0 and 2 to the next row, then lane
    31 to the upper half."""
    for shift in (1, 2, 4, 8):
        v = [f32(v[l - shift] + v[l]) if l & 15 >= shift else v[l] for l in range(64)]
    v = [f32(v[(l & ~15) - 1] + v[l]) if l >> 4 in (1, 3) else v[l] for l in range(64)]
    return [f32(v[31] + v[l]) if l >= 32 else v[l] for l in range(64)]


def binade(x):
    return int(f32(x).view(np.int32)) >> 23


def chain(addends, acc):
    for x in addends:
        acc = f32(acc + x)
    return acc


def guess_misses(squares):
    """(whether a leap starts or ends in another binade than its guess, how many parts are walked by themselves, the sum, what
    the leaps alone would have made of it)"""
    words = (len(squares) + 1023) >> 10
    addends = np.zeros(1024 * words, f32)
    addends[:len(squares)] = squares
    parts = addends.reshape(64, 4, words, 4)
    sums, total = np.zeros((64, 4), f32), np.zeros(64, f32)
    for p in range(4):
        for w in range(words):
            v = parts[:, p, w]
            sums[:, p] += (v[:, 0] + v[:, 1]) + (v[:, 2] + v[:, 3])
        total += sums[:, p]
    guess = np.array([0.0] + scan(total)[:-1], f32)
    starts = np.zeros((64, 4), f32)
    for p in range(4):
        starts[:, p] = guess
        guess = guess + sums[:, p]
    missed, walked, before, acc, leapt = False, 0, -1, f32(0), f32(0)
    for start, part in zip(starts.reshape(-1), addends.reshape(256, -1)):
        even = int(start.view(np.int32)) & ~1
        here = even >> 23
        ends = [int(chain(part, np.int32(s).view(f32)).view(np.int32)) for s in (even, even | 1)]
        stays = all(end >> 23 == here for end in ends)
        cut = not stays or (before >= 0 and before != here)
        after = chain(part, acc)
        if cut:
            walked += 1
            leapt = chain(part, leapt)
        else:
            missed = missed or binade(acc) != here or binade(after) != here
            bits = int(leapt.view(np.int32))
            leapt = np.int32(bits + ends[bits & 1] - (even | bits & 1)).view(f32)
        before, acc = here if stays else -1, after
    return missed, walked, acc, leapt


@pytest.mark.parametrize("n", [1025, 2047, 2049, 2816, 3072, 3073, 4095, 4096])
@pytest.mark.parametrize("kind", ["stagnant", "overtaking"])
def test_a_chain_that_misses_its_guess(kind, n):
    x = vector(kind, n, cases.synth.rng(1))
    missed, _, total, leapt = guess_misses(x * x)
    assert missed or (kind == "stagnant" and n < 2047)
    assert leapt != total or kind == "stagnant"         # where the guess matters, the leaps alone give another sum


@pytest.mark.parametrize("n", [768, 2816, 4096])
def test_ordinary_vectors_are_guessed(n):
    x = vector("normal", n, cases.synth.rng(n))
    missed, walked, total, leapt = guess_misses(x * x)
    assert not missed and walked < 40 and leapt == total
