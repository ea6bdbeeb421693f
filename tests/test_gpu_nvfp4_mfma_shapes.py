"""Prefill-sized NVFP4 matmul: both tile forms, columns split over workgroups and not, fewer stages than a chunk of codes,
ragged tiles, and block scales on an odd pair of bytes (fetched two bytes at a time instead of sixteen).  Sampled rows
against the CPU checker with the bound of the entry point, 2^-20 * sum_c |w_c x_c|."""
import numpy as np
import pytest

from golden import cases
from test_gpu_nvfp4_mfma import reference

pytestmark = pytest.mark.gpu
synth = cases.synth


@pytest.mark.parametrize("R,C,B,offset", [
    (130, 128, 65, 0), (257, 192, 33, 2), (70, 576, 64, 0), (200, 4096, 40, 2),     # 64 x 128 tiles, one to eight splits
    (8200, 512, 129, 0), (8200, 1088, 70, 2),                                       # one split
    (27400, 64, 130, 0), (27400, 320, 130, 0), (27400, 320, 130, 2),                # 64 x 256 tiles
])
def test_tile_forms(pkg, oracle, R, C, B, offset):
    print(f"nvfp4 mfma forms R={R} C={C} B={B} offset={offset}", flush=True)
    gpu = pkg.lib
    lib = gpu.init()
    packed, scales = synth.nvfp4_tensor(R, C, R + C)
    xs = synth.activations(C, B, 41)
    dp, dx, dy = gpu.DeviceBuffer.from_host(packed), gpu.DeviceBuffer.from_host(xs), gpu.DeviceBuffer(B * R * 4, fill=0xFF)
    ds, status = gpu.DeviceBuffer(scales.nbytes + offset), gpu.DeviceBuffer(4, fill=0x7F)
    ds.upload(scales, offset)
    ws = gpu.DeviceBuffer(lib.salt_mi355_nvfp4_matmul_workspace_bytes(R, C, B))
    stream = lib.salt_mi355_stream()
    gpu.check(lib.salt_mi355_nvfp4_matmul_dev(dp.ptr, ds.ptr + offset, 2688.0, 64.0, R, C, B, dx.ptr, dy.ptr, status.ptr, ws.ptr,
                                              stream), "nvfp4_matmul_dev")
    gpu.check(lib.salt_mi355_stream_sync(stream), "sync")
    got = dy.to_host(np.float32).reshape(B, R)
    assert status.to_host(np.int32)[0] == 0 and np.isfinite(got).all()
    rows = np.unique(np.r_[np.arange(0, R, max(1, R // 60)), R - 1])
    sub_packed = np.ascontiguousarray(packed.reshape(R, C // 2)[rows]).reshape(-1)
    sub_scales = np.ascontiguousarray(scales.reshape(R, C // 16)[rows]).reshape(-1)
    want, mags = reference(oracle, sub_packed, sub_scales, 2688.0, 64.0, len(rows), C, xs)
    ratio = float((np.abs(got[:, rows].astype(np.float64) - want) / (2.0 ** -20 * mags + 1e-30)).max())
    print("max err / bound", ratio, flush=True)
    assert ratio <= 1.0
