"""The sum of squares of a norm is the left-to-right fp32 chain whatever its values do to the accumulator: ties to even,
jumps over many powers of two, subnormals, overflow, sizes around every layout's edge."""
import ctypes as C

import numpy as np
import pytest

from golden import cases
from oracle_lib import bits, ffn_layer_struct, host_threads, ptr

pytestmark = pytest.mark.gpu
synth = cases.synth
f32 = np.float32


@pytest.fixture(scope="module")
def gpu(pkg):
    pkg.lib.init()
    return pkg.lib


def vector(kind, n, g):
    x = g.standard_normal(n)
    if kind == "ties":                      # the first square is 2^12 (unit 2^-11), every other one an odd multiple of 2^-12
        x = (2 * g.integers(0, 40, n) + 1) * 2.0 ** -6
        x[0] = 64.0
    elif kind == "ones":
        x = np.ones(n)
        x[0] = 4096.0                       # a unit of two
    elif kind == "growing":
        x = x * np.exp2(np.linspace(-40, 40, n))
    elif kind == "falling":
        x = x * np.exp2(np.linspace(40, -40, n))
    elif kind == "outliers":
        x = np.where(g.random(n) < 0.004, 1e3 * x, 1e-3 * x)
    elif kind == "zeros":
        x = np.where(np.arange(n) == n * 2 // 3, 0.75, 0.0)
    elif kind == "subnormal":
        x = x * 3e-22
    elif kind == "edge":                    # the sum passes a power of two at almost every boundary between parts
        x = np.where(np.arange(n) % 12 == 11, np.sqrt(np.exp2(np.arange(n) // 48 - 20.0)), 1e-4 * x)
    elif kind == "overflow":
        x = x * 1e18
    elif kind == "stagnant":                # squares of less than half a unit leave the chain below two, a plain sum passes it
        x = np.full(n, 2.0 ** -12.5)
        x[0] = np.sqrt(2 - 2.0 ** -15)
    elif kind == "overtaking":              # squares that the chain rounds up to a unit each: it passes two before a plain sum
        x = np.full(n, np.sqrt(0.6) * 2.0 ** -11.5)
        x[0] = np.sqrt(2 - 200 * 2.0 ** -23)
    return x.astype(f32)


KINDS = ["normal", "ties", "ones", "growing", "falling", "outliers", "zeros", "subnormal", "edge", "overflow", "stagnant", "overtaking"]


@pytest.mark.parametrize("n", [1, 2, 3, 5, 31, 33, 64, 511, 512, 513, 735, 736, 737, 1024, 1025, 2047, 2049, 2816, 3072, 3073, 4095, 4096, 4097, 4608, 9000])
def test_sum_of_squares_is_the_chain(gpu, oracle, n):
    eps = f32(1e-6)
    for at, kind in enumerate(KINDS):
        print("ordered sum", n, kind, flush=True)
        g = synth.rng(1000 * n + at)
        x, dense, routed, res = (vector(kind, n, g) for _ in range(4))
        w = (1.0 + 0.1 * g.standard_normal(n)).astype(f32)
        want = np.full(n, np.nan, f32)
        rc = oracle.orc_rmsnorm(ptr(want), ptr(x), ptr(w), n, eps, 1)
        st, got = gpu.run_cells([(gpu.CELL_RMSNORM, ["x", "w", "out"], n, 1, eps, 0.0)],
                                {"x": x, "w": w, "out": np.full(n, np.nan, f32)})
        assert st == rc
        if rc == 0:
            assert np.array_equal(bits(got["out"]), bits(want))
        want = np.full(n, np.nan, f32)
        rc = oracle.orc_parallel_ffn_combine(ptr(want), ptr(res), ptr(dense), ptr(routed), ptr(w), ptr(w), ptr(w), f32(0.37), n,
                                             eps)
        arrays = {"res": res, "dense": dense, "routed": routed, "w": w, "scratch": np.zeros(2 * n, f32),
                  "out": np.full(n, np.nan, f32)}
        st, got = gpu.run_cells([(gpu.CELL_PARALLEL_COMBINE, ["res", "dense", "routed", "w", "w", "w", "scratch", "out"], n, 0,
                                  eps, 0.37)], arrays)
        assert st == rc
        if rc == 0:
            assert np.array_equal(bits(got["out"]), bits(want))


@pytest.mark.parametrize("H", [704, 768, 2816, 4096, 4160])
def test_first_norm_of_a_block(gpu, oracle, H):
    """The same vectors as the residual of a feed-forward block, whose first launch has a kernel of its own."""
    D, F, E, K = 64, 64, 2, 1
    w = synth.ffn_layer(H, D, F, E, K, 3)
    block, layer = gpu.FfnBlock(w), ffn_layer_struct(w)
    for at, kind in enumerate(KINDS):
        print("ordered sum, block", H, kind, flush=True)
        residual = vector(kind, H, synth.rng(50 * H + at))
        want, sel, wt = np.zeros(H, f32), np.zeros(K, np.int32), np.zeros(K, f32)
        rc = oracle.orc_ffn_block(C.byref(layer), ptr(residual), ptr(want), ptr(sel), ptr(wt), host_threads())
        st, gsel, gwt, out = block.step(residual)
        assert st == rc
        if rc == 0:
            assert np.array_equal(gsel, sel) and np.array_equal(bits(gwt), bits(wt)) and np.array_equal(bits(out), bits(want))
