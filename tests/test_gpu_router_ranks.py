"""The router's ranks at the edges of its batches of four and sixteen logits and of its parts of a workgroup, among equal
logits and both zeros: alone (one part) and inside the exact MoE step, whose workgroups of 512 threads spread the comparisons of
few experts over up to eight parts.  Bit-for-bit against the CPU checker."""
import ctypes as ct

import numpy as np
import pytest

from golden import cases
from oracle_lib import ExpertGeometry, bits, ptr

pytestmark = pytest.mark.gpu
synth = cases.synth


def logits_of(kind, E, g):
    x = g.standard_normal(E).astype(np.float32)
    if kind == "ties": x = (np.round(x * 2) / 2).astype(np.float32)
    if kind == "equal": x = np.where(g.random(E) < 0.5, np.float32(0.0), np.float32(-0.0))
    return x


@pytest.mark.parametrize("E", [1, 3, 4, 5, 15, 16, 17, 63, 64, 65, 127, 128, 129, 192, 255, 256, 257, 300, 511, 512, 1000, 1024])
def test_ranks_at_every_edge(pkg, oracle, E):
    gpu = pkg.lib
    gpu.init()
    H = F = 64
    pool = np.tile(synth.expert_pool(min(E, 8), H, F, 1).reshape(min(E, 8), -1), (-(-E // 8), 1))[:E].reshape(-1)
    for at, kind in enumerate(["normal", "ties", "equal"]):
        g = synth.rng(10 * E + at)
        K = min(E, int(g.integers(1, 9)))
        logits, scale = logits_of(kind, E, g), g.uniform(0.25, 4, E).astype(np.float32)
        print("router ranks", E, K, kind, flush=True)
        sel, w = np.zeros(K, np.int32), np.zeros(K, np.float32)
        assert oracle.orc_router_topk(ptr(logits), ptr(scale), E, K, ptr(sel), ptr(w)) == 0
        st, gsel, gw = gpu.router_topk(logits, scale, K)
        assert st == 0 and np.array_equal(gsel, sel) and np.array_equal(bits(gw), bits(w))
        if E > 512:
            continue
        x = synth.activations(H, 1, at)[0]
        status, gsel, gw, eo, y = gpu.MoeLayer(pool, E, H, F, K).step(logits, scale, x)
        osel, ow, oeo, oy = np.zeros(K, np.int32), np.zeros(K, np.float32), np.zeros((K, H), np.float32), np.zeros(H, np.float32)
        assert oracle.orc_moe_decode_step(ct.byref(ExpertGeometry(H, F)), ptr(pool), E, K, ptr(logits), ptr(scale), ptr(x),
                                          ptr(osel), ptr(ow), ptr(oeo), ptr(oy), 2) == 0
        assert status == 0 and np.array_equal(gsel, osel) and np.array_equal(bits(gw), bits(ow))
        assert np.array_equal(bits(eo), bits(oeo)) and np.array_equal(bits(y), bits(oy))


@pytest.mark.parametrize("E,K", [(5, 5), (64, 64), (300, 64)])
def test_weights_of_a_whole_wave(pkg, oracle, E, K):
    g = synth.rng(E)
    logits, scale = (3 * g.standard_normal(E)).astype(np.float32), g.uniform(0.25, 4, E).astype(np.float32)
    sel, w = np.zeros(K, np.int32), np.zeros(K, np.float32)
    assert oracle.orc_router_topk(ptr(logits), ptr(scale), E, K, ptr(sel), ptr(w)) == 0
    st, gsel, gw = pkg.lib.router_topk(logits, scale, K)
    assert st == 0 and np.array_equal(gsel, sel) and np.array_equal(bits(gw), bits(w))
