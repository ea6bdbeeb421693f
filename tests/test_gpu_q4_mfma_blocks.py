"""Blocks of 64 and of 32 tokens in one launch of the prefill matmul: the limits of the rule for one matrix, the last block
of one token, and experts whose numbers of tokens lie around both block sizes.

A token's bits do not depend on the block that holds it, so calls small enough for one kind of block are the reference for
the mixture; their own values have the entry point's bound elsewhere."""
import ctypes as C

import numpy as np
import pytest

from golden import cases
from moe_bounds import group_term_magnitudes
from oracle_lib import ExpertGeometry, host_threads, ptr
from test_gpu_moe_prefill import check_values, expected_grouping
from test_gpu_q4_mfma_shapes import check, name_of

pytestmark = pytest.mark.gpu
synth = cases.synth


@pytest.mark.parametrize("R,C_,B,form", [
    (16640, 128, 257, (3, 3)),          # 65 tiles of rows, nine halves: a last block of one token
    (16384, 192, 288, (4, 1)),          # 576 halves, four blocks of 64 as there would be anyway
    (16380, 128, 383, (4, 4)),          # 768, the upper limit
    (16384, 128, 416, (6, 1)),          # 832, past it
    (4000, 128, 1057, (16, 2)),         # 16 tiles of rows, 544 halves
    (33000, 64, 150, (2, 1)),           # 129 tiles of rows: 516 tiles with one block of 64, too many
    (32700, 64, 190, (2, 2)),           # 128 and 768
    (65700, 64, 70, (1, 1)),            # 257: more than compute units, and 771 halves
    (65500, 64, 96, (1, 1)),            # 256 and 768
])
def test_mixed_blocks(pkg, oracle, R, C_, B, form):
    print(f"mfma blocks R={R} C={C_} B={B}", flush=True)
    vals, scales, biases = synth.q4_tensor(R, C_, R + B)
    xs = synth.activations(C_, B, 31)
    got = pkg.lib.q4_matmul(vals, scales, biases, R, C_, xs).view(np.uint32)
    assert pkg.lib.load().salt_mi355_last_kernel().decode() == name_of(*form)
    step = 32 * max(1, 256 // -(-R // 256))
    for first in range(0, B, step):
        piece = pkg.lib.q4_matmul(vals, scales, biases, R, C_, xs[first:first + step])
        assert np.array_equal(piece.view(np.uint32), got[first:first + step]), first
    rows = 64                                                   # and these against the reference
    check(pkg, oracle, vals[:rows * C_ // 8], scales[:rows * C_ // 64], biases[:rows * C_ // 64], rows, C_, xs[:70])


EDGES = [0, 1, 31, 32, 33, 0, 63, 64, 65, 95, 96, 97, 128, 129, 0]
LONG = [33, 65568, 0, 40]               # one expert with 1025 blocks of 64 tokens, more than a workgroup has threads


@pytest.mark.parametrize("H,F,counts", [(128, 320, EDGES), (320, 128, EDGES), (64, 64, LONG)])
def test_experts_around_the_block_sizes(pkg, oracle, H, F, counts):
    print(f"prefill blocks H={H} F={F}", flush=True)
    E, T, K = len(counts), sum(counts), 1
    sel = np.random.default_rng(3).permutation(np.repeat(np.arange(E, dtype=np.int32), counts)).reshape(T, K)
    w = np.ones((T, K), np.float32)
    pool, xs = synth.expert_pool(E, H, F, 4), synth.activations(H, T, 5)
    want = np.zeros((T, H), np.float32)
    g = ExpertGeometry(H, F)
    assert oracle.orc_moe_group(C.byref(g), ptr(pool), E, K, T, ptr(sel), ptr(w), ptr(xs), ptr(want), None, host_threads()) == 0
    layer = pkg.lib.MoePrefill(pool, E, H, F, K, T)
    status, ys, rows, pairs = layer.run(sel, w, xs)
    want_rows, want_pairs = expected_grouping(sel, E)
    assert status == 0 and np.array_equal(rows, want_rows) and np.array_equal(pairs, want_pairs)
    check_values(ys, want, group_term_magnitudes(pool, sel, w, xs, H, F))
