"""Device memory helpers: a fill is done when it returns, also for work on a stream that does not wait for the null stream."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_a_launch_after_a_fill_is_not_overwritten_by_it(pkg):
    """A kernel that writes the last kilobyte of a large buffer right after the buffer's fill."""
    gpu = pkg.lib
    lib = gpu.init()
    stream = lib.salt_mi355_stream()
    size = 4 << 30
    buf = gpu.DeviceBuffer(size)
    at = size - 1024

    def write():
        gpu.check(lib.salt_mi355_router_fixture_dev(128, 8, 5, 3, 0.5, buf.at(at), buf.at(at + 512), stream), "fixture router")

    def read():
        gpu.check(lib.salt_mi355_stream_sync(stream), "sync")
        return buf.to_host(np.int32, 8, at), buf.to_host(np.float32, 8, at + 512)

    write()
    want = read()
    assert sorted(set(want[0])) == sorted(want[0]) and (want[1] > 0).all()
    for value in (0x00, 0xFF, 0x11):
        print("fill", value, flush=True)
        gpu.check(lib.salt_mi355_dev_fill(buf.ptr, value, size), "fill")
        write()
        idx, w = read()
        assert np.array_equal(idx, want[0]) and np.array_equal(w, want[1])
        gap = buf.to_host(np.uint8, 256, at + 256)
        assert (gap == value).all()
