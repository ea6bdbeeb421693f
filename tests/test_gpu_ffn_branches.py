"""The feed-forward block with both branches in the same launches, at every shape that its routed gate/up launch can take, and
at the limits beyond which the dense branch runs on the second stream: bit-for-bit against the CPU checker."""
import ctypes as C

import numpy as np
import pytest

from golden import cases
from oracle_lib import bits, ffn_layer_struct, host_threads, ptr

pytestmark = pytest.mark.gpu
synth = cases.synth
f32 = np.float32


def together(gate_up, down):
    """What a block reports whose branches share their launches."""
    return f"ffn_gate_kernel + q4_tile_kernel<{gate_up}> + ffn_down_kernel<{down}>"


SECOND_STREAM = "q4_tile_kernel<2,1,32,0>"          # the dense down projection by itself, in whole tiles


@pytest.mark.parametrize("H,D,F,E,K,launches", [
    (64, 64, 64, 1, 1, together("2,1,32,1,2", "1,32,4")),
    (1088, 1024, 576, 16, 1, together("2,1,32,1,2", "1,32,4")),         # 18 tiles: halves; down 17: quarters, one chain per lane
    (2112, 1216, 1024, 32, 2, together("1,1,32,1,4", "2,32,2")),        # 64: quarters, one chain per lane
    (1280, 4096, 640, 16, 8, together("2,1,16,1,4", "2,32,1")),         # 160: quarters; the widest dense branch; down 160: whole
    (1024, 128, 640, 16, 8, together("2,1,16,1,4", "2,32,2")),          # 160; down 128: halves
    (1920, 704, 1216, 20, 6, together("4,1,16,1,2", "2,32,1")),         # 228: halves, four chains
    (512, 320, 1600, 24, 8, together("4,1,16,1,1", "1,32,4")),          # 400: whole tiles, four chains
    (512, 192, 640, 300, 8, together("2,1,32,1,1", "1,32,4")),          # more than 256 experts: whole
    (4096, 192, 64, 8, 2, together("1,1,32,1,4", "2,32,2")),            # the widest gate
    (256, 4160, 128, 16, 4, SECOND_STREAM),                             # a dense branch too wide
    (4160, 192, 64, 8, 2, SECOND_STREAM),                               # a gate too wide
])
def test_block_matches_the_checker(pkg, oracle, H, D, F, E, K, launches):
    print("ffn branches", H, D, F, E, K, flush=True)
    pkg.lib.init()
    w = synth.ffn_layer(H, D, F, E, K, 21)
    block = pkg.lib.FfnBlock(w)
    layer = ffn_layer_struct(w)
    want, osel, owt = np.zeros(H, f32), np.zeros(K, np.int32), np.zeros(K, f32)
    for seed in (31, 32):
        residual = (synth.activations(H, 1, seed)[0] * 3).astype(f32)
        st, sel, wt, out = block.step(residual)
        assert pkg.lib.load().salt_mi355_last_kernel().decode() == launches
        assert oracle.orc_ffn_block(C.byref(layer), ptr(residual), ptr(want), ptr(osel), ptr(owt), host_threads()) == 0
        assert st == 0 and np.array_equal(sel, osel) and np.array_equal(bits(wt), bits(owt)) and np.array_equal(bits(out), bits(want))
    residual[H // 2] = np.nan
    st, _, _, kept = block.step(residual)
    assert st == -1 and np.array_equal(bits(kept), bits(out))
