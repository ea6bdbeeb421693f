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
    """The expected form: 64 x 256 tiles from 320 of them on; else 64 x 128 and the columns split over workgroups while each
    still has a compute unit, eight chunks of 64 columns at least per split."""
    wide = -(-B // 64) * -(-R // 256) >= 320
    split = 1 if wide else max(1, min(256 // (-(-B // 64) * -(-R // 128)), 8, C // 64 // 8))
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
    form, _, splits = lib.salt_mi355_last_kernel().decode().rpartition(" ksplit ")
    assert form == ("fp4_mfma_kernel<4,4,0>" if wide else "fp4_mfma_kernel<8,2,0>")
    assert int(splits) == split
    assert status.to_host(np.int32)[0] == 0 and np.isfinite(got).all()
    rows = np.unique(np.r_[np.arange(0, R, max(1, R // 60)), R - 1])
    sub_packed = np.ascontiguousarray(packed.reshape(R, C // 2)[rows]).reshape(-1)
    sub_scales = np.ascontiguousarray(scales.reshape(R, C // 16)[rows]).reshape(-1)
    want, mags = reference(oracle, sub_packed, sub_scales, 2688.0, 64.0, len(rows), C, xs)
    ratio = float((np.abs(got[:, rows].astype(np.float64) - want) / (2.0 ** -20 * mags + 1e-30)).max())
    print("max err / bound", ratio, flush=True)
    assert ratio <= 1.0


def test_rows_beyond_32_bit_offsets(pkg, oracle):
    """33 554 496 columns: the offset of the last of 64 token rows passes 2^32 bytes, that of a second weight row 2^24.
    All tokens but the first and the last are zero."""
    R, C, B = 2, (1 << 25) + 64, 64
    print(f"nvfp4 mfma far rows C={C}", flush=True)
    gpu = pkg.lib
    lib = gpu.init()
    packed, scales = synth.nvfp4_tensor(R, C, 3)
    ends = synth.activations(C, 2, 5)
    dp, ds, dx = gpu.DeviceBuffer.from_host(packed), gpu.DeviceBuffer.from_host(scales), gpu.DeviceBuffer(4 * B * C, fill=0)
    dx.upload(ends[0])
    dx.upload(ends[1], 4 * (B - 1) * C)
    dy, status = gpu.DeviceBuffer(B * R * 4, fill=0xFF), gpu.DeviceBuffer(4, fill=0x7F)
    ws = gpu.DeviceBuffer(lib.salt_mi355_nvfp4_matmul_workspace_bytes(R, C, B))
    stream = lib.salt_mi355_stream()
    gpu.check(lib.salt_mi355_nvfp4_matmul_dev(dp.ptr, ds.ptr, 2688.0, 64.0, R, C, B, dx.ptr, dy.ptr, status.ptr, ws.ptr, stream),
              "nvfp4_matmul_dev")
    gpu.check(lib.salt_mi355_stream_sync(stream), "sync")
    got = dy.to_host(np.float32).reshape(B, R)
    assert lib.salt_mi355_last_kernel().decode() == "fp4_mfma_kernel<8,2,1> ksplit 8"
    assert status.to_host(np.int32)[0] == 0 and (got[1:-1] == 0).all()
    want, mags = reference(oracle, packed, scales, 2688.0, 64.0, R, C, ends)
    ratio = float((np.abs(got[[0, -1]].astype(np.float64) - want) / (2.0 ** -20 * mags)).max())
    print("max err / bound", ratio, flush=True)
    assert ratio <= 1.0
