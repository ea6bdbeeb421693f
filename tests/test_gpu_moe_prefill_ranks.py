"""Grouped prefill: more than eight experts per token (the selection is then checked from memory), and tokens whose bits do
not depend on the tokens they come with where one call would fill the device and another would not."""
import numpy as np
import pytest

import test_gpu_moe_prefill as base

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
