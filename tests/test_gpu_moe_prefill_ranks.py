"""Grouped prefill: more than eight experts per token (the selection is then checked from memory); tokens whose bits do not
depend on the tokens they come with, from a call that fills the device to one of a few tokens; scales too far apart for
one fp16 operand range."""
import ctypes as ct

import numpy as np
import pytest

import test_gpu_moe_prefill as base
from oracle_lib import ExpertGeometry, host_threads, ptr

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,K,H,F", [(70, 20, 9, 128, 64), (33, 16, 16, 64, 128), (300, 16, 2, 1024, 512)])
def test_many_ranks_and_token_independence(pkg, oracle, T, E, K, H, F):
    base.test_against_cpu_checker(pkg, oracle, T, E, K, H, F)


@pytest.mark.parametrize("kind", ["duplicate", "range", "nan"])
def test_invalid_selection_of_many_ranks(pkg, kind):
    T, E, K, H, F = 70, 20, 9, 128, 64
    print("prefill invalid", kind, flush=True)
    synth = base.synth
    layer = pkg.lib.MoePrefill(synth.expert_pool(E, H, F, 5), E, H, F, K, T)
    sel, w = synth.zipf_selection(T, E, K, 1.1, 6)
    sel, w = sel.copy(), w.copy()
    if kind == "duplicate": sel[69, 8] = sel[69, 0]
    if kind == "range": sel[64, 8] = E
    if kind == "nan": w[3, 8] = np.nan
    status, ys, _, _ = layer.run(sel, w, synth.activations(H, T, 7))
    assert status == -1 and (ys.view(np.uint32) == 0xFFFFFFFF).all()


@pytest.mark.parametrize("T,E,K,H,F", [(1200, 16, 2, 1024, 512), (300, 16, 2, 1024, 512), (600, 8, 3, 1088, 704)])
def test_prefixes_have_the_bits_of_the_whole(pkg, T, E, K, H, F):
    """Calls of 1, 3, 20 and 150 tokens have a few to a hundred tiles per launch, the whole one two to six hundred."""
    print("prefill prefixes", T, E, K, H, F, flush=True)
    synth = base.synth
    layer = pkg.lib.MoePrefill(synth.expert_pool(E, H, F, 5), E, H, F, K, T)
    sel, w = synth.zipf_selection(T, E, K, 1.1, 6)
    xs = synth.activations(H, T, 7)
    status, whole, _, _ = layer.run(sel, w, xs)
    assert status == 0
    for n in (1, 3, 20, 150):
        status, part, _, _ = layer.run(sel[:n], w[:n], xs[:n])
        assert status == 0 and np.array_equal(part.view(np.uint32), whole[:n].view(np.uint32)), n


def test_scales_far_apart(pkg, oracle):
    """Gate and up groups of 2^40 that meet zeros beside the ordinary ones: tiles of 64 and fewer tokens walk their columns
    more than once."""
    T, E, K, H, F = 300, 4, 2, 640, 128
    print("prefill windows", flush=True)
    synth = base.synth
    pool = synth.expert_pool(E, H, F, 8)
    far = np.arange(H // 64) % 3 == 1
    proj, n = synth.expert_proj_bytes(H, F), H * F
    for e in range(E):
        for p in range(2):
            at = (e * 3 + p) * proj + n // 2
            pool[at:at + n // 32].view(np.uint16).reshape(F, -1)[:, far] = 0x5380              # 2^40
            pool[at + n // 32:at + n // 16].view(np.uint16).reshape(F, -1)[:, far] = 0xD4F0    # -7.5 times that
    sel, w = synth.zipf_selection(T, E, K, 1.1, 9)
    xs = synth.activations(H, T, 10)
    xs[:, np.repeat(far, 64)] = 0.0
    want = np.zeros((T, H), np.float32)
    assert oracle.orc_moe_group(ct.byref(ExpertGeometry(H, F)), ptr(pool), E, K, T, ptr(sel), ptr(w), ptr(xs), ptr(want), None,
                                host_threads()) == 0
    status, ys, _, _ = pkg.lib.MoePrefill(pool, E, H, F, K, T).run(sel, w, xs)
    assert status == 0
    base.check_values(ys, want, base.term_magnitudes(pool, sel, w, xs, H, F))
