"""NVFP4 activation pass at the edges of its grid: remainders of a workgroup's 256 blocks, and more blocks than one grid
dimension has threads for (2^32 threads, four per block)."""
import numpy as np
import pytest

from golden import cases
from oracle_lib import bits, ptr

pytestmark = pytest.mark.gpu
synth = cases.synth


def expected(oracle, x, g):
    C = x.size
    packed, scales, dequant = np.zeros(C // 2, np.uint8), np.zeros(C // 16, np.uint8), np.zeros(C, np.float32)
    assert oracle.orc_nvfp4_qdq(ptr(x), C, g, ptr(packed), ptr(scales), ptr(dequant)) == 0
    return packed, scales, dequant


@pytest.mark.parametrize("C,B,filled", [(16, 1, None), (4080, 1, None), (4096, 1, None), (4112, 3, None),
                                        (1 << 16, (1 << 14) + 1, 4), (1 << 16, (1 << 18) + 1, 3)])
def test_grid_edges(pkg, oracle, C, B, filled):
    """`filled` tokens at the start, the middle and the end hold values, the others zeros."""
    print(f"qdq C={C} B={B}", flush=True)
    gpu, g = pkg.lib, 64.0
    lib = gpu.init()
    stream = lib.salt_mi355_stream()
    tokens = range(B) if filled is None else sorted({0, B // 2, B - 1, *range(filled - 3)})
    xs = synth.activations(C, len(tokens), C + B)
    dx, dd = gpu.DeviceBuffer(4 * B * C, fill=0), gpu.DeviceBuffer(4 * B * C)
    dp, ds, status = gpu.DeviceBuffer(B * C // 2), gpu.DeviceBuffer(B * C // 16, fill=0xFF), gpu.DeviceBuffer(4, fill=0)
    for t, x in zip(tokens, xs):
        dx.upload(x, 4 * t * C)
    gpu.check(lib.salt_mi355_nvfp4_qdq_dev(dx.ptr, C, B, g, dp.ptr, ds.ptr, dd.ptr, status.ptr, stream), "nvfp4_qdq_dev")
    gpu.check(lib.salt_mi355_stream_sync(stream), "sync")
    assert status.to_host(np.int32)[0] == 0
    scales = ds.to_host(np.uint8).reshape(B, C // 16)
    for t, x in zip(tokens, xs):
        packed, want_scales, dequant = expected(oracle, x, g)
        assert np.array_equal(scales[t], want_scales), t
        assert np.array_equal(dp.to_host(np.uint8, C // 2, t * (C // 2)), packed), t
        # zeros differ in sign: the reference's index of a zero is the lowest
        assert np.array_equal(dd.to_host(np.float32, C, 4 * t * C), dequant), t
    assert not np.delete(scales, list(tokens), axis=0).any()
