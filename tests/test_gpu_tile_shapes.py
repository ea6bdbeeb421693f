"""Every shape that a launch of the bit-exact Q4 kernel can take by its number of tiles, tokens and columns, pinned by name, with
ragged last tiles and a scale that the converter's power of two overflows; the MoE step's launches in parts of tiles."""
import ctypes as ct

import numpy as np
import pytest

from golden import cases
from oracle_lib import ExpertGeometry, bits, host_threads, ptr

pytestmark = pytest.mark.gpu
synth = cases.synth

# rows of the jobs, columns, tokens, kernel
SHAPES = [
    ((70, 1, 1033, 333), 1088, (1,), "q4_tile_kernel<1,1,32,0,4>"),                      # 25 tiles
    ((4096,), 1024, (1,), "q4_tile_kernel<1,1,32,0,4>"),                                 # 64 tiles
    ((4096,), 960, (1,), "q4_tile_kernel<2,1,32,0,4>"),
    ((2112, 2049, 7), 1216, (1,), "q4_tile_kernel<1,1,32,0,8>"),                         # 67 tiles
    ((6143,), 1024, (1,), "q4_tile_kernel<1,1,32,0,8>"),                                 # 96 tiles
    ((6143,), 128, (1,), "q4_tile_kernel<2,1,32,0,4>"),
    ((6145,), 1024, (1,), "q4_tile_kernel<2,1,32,0,2>"),                                 # 97 tiles
    ((8193,), 576, (1,), "q4_tile_kernel<2,1,16,0,4>"),                                  # 129 tiles
    ((4096, 4095, 4033), 1088, (1,), "q4_tile_kernel<2,1,16,0,4>"),                      # 192 tiles
    ((12289,), 192, (1,), "q4_tile_kernel<2,1,16,0,2>"),                                 # 193 tiles
    ((16384,), 64, (1,), "q4_tile_kernel<2,1,16,0,2>"),                                  # 256 tiles
    ((8000,), 8256, (1,), "q4_tile_kernel<2,1,32,0>"),                                   # too wide a row for parts
    ((70, 1, 1033, 333), 1088, (2, 3, 4), "q4_tile_kernel<1,{},16,0,4>"),
    ((17, 31), 8256, (2, 3, 4), "q4_tile_kernel<1,{},16,0,4>"),
    ((2112, 2049, 7), 576, (2, 3, 4), "q4_tile_kernel<2,{},16,0,2>"),
    ((8193,), 576, (2, 3, 4), "q4_tile_kernel<2,{},16,0,4>"),
    ((12289,), 192, (2, 3, 4), "q4_tile_kernel<2,{},16,0,2>"),
    ((32769,), 192, (2, 3, 4), "q4_tile_kernel<4,{},16,0,2>"),                           # 513 tiles
    ((40960,), 64, (2, 3, 4), "q4_tile_kernel<4,{},16,0,2>"),                            # 640 tiles
    ((40961,), 64, (2, 3, 4), "q4_tile_kernel<4,{},16,0>"),
    ((32769,), 64, (1,), "q4_tile_kernel<4,1,16,0>"),
]


# the same where the caller states the chains per lane: whole tiles
STATED = [
    ((70, 1, 1033, 333), 1088, (1,), 4, "q4_tile_kernel<4,1,16,0>"),                     # 25 tiles
    ((16384,), 64, (1,), 4, "q4_tile_kernel<4,1,16,0>"),                                 # 256
    ((16385,), 64, (1, 2, 3, 4), 4, "q4_tile_kernel<4,{},16,0>"),
    ((70, 1033), 1088, (1,), 2, "q4_tile_kernel<2,1,32,0>"),
    ((16385,), 64, (1, 2, 3, 4), 2, "q4_tile_kernel<2,{},16,0>"),
    ((70, 1033), 1088, (1, 2, 3, 4), 8, "q4_tile_kernel<8,{},16,0>"),
]


@pytest.mark.parametrize("rows,C,tokens,chains,kernel", [(r, c, t, 0, k) for r, c, ts, k in SHAPES for t in ts] +
                         [(r, c, t, n, k) for r, c, ts, n, k in STATED for t in ts])
def test_every_shape(pkg, oracle, rows, C, tokens, chains, kernel):
    print(f"q4 shape {kernel} rows={rows} C={C} tokens={tokens} chains={chains}", flush=True)
    lib = pkg.lib.init()
    stream = lib.salt_mi355_stream()
    hold, jobs, want = [], (pkg.lib.Q4Job * len(rows))(), []
    for j, R in enumerate(rows):
        vals, scales, biases = synth.q4_tensor(R, C, 70 + j)
        if j == 1:
            scales = scales.copy()
            scales[-1] = 0x7B80                  # 2^120, in the job's last row
        xs = synth.activations(C, tokens, 80 + j)
        y = np.zeros((tokens, R), np.float32)
        for t in range(tokens):
            assert oracle.orc_q4_matvec_threads(ptr(vals), ptr(scales), ptr(biases), R, C, ptr(xs[t]), ptr(y[t]), host_threads()) == 0
        bufs = [pkg.lib.DeviceBuffer.from_host(a) for a in (vals, scales, biases, xs)] + [pkg.lib.DeviceBuffer(y.nbytes, fill=0xFF)]
        jobs[j] = pkg.lib.Q4Job(*[b.ptr for b in bufs], R)
        hold.append(bufs)
        want.append(y)
    pkg.lib.check(lib.salt_mi355_q4_jobs_dev(jobs, len(rows), C, tokens, chains, stream), "q4_jobs_dev")
    pkg.lib.check(lib.salt_mi355_stream_sync(stream), "sync")
    assert lib.salt_mi355_last_kernel().decode() == kernel.format(tokens)
    for bufs, y in zip(hold, want):
        assert np.array_equal(bits(bufs[4].to_host(np.float32).reshape(y.shape)), bits(y))


@pytest.mark.parametrize("E,K,H,F,gate_up,down", [
    (16, 1, 1088, 576, "2,1,32,1,2", "1,1,32,2,4"),      # gate/up 18 tiles: halves; down 17: quarters
    (32, 2, 2112, 1024, "1,1,32,1,4", "2,1,32,2,2"),     # 64: quarters with one chain; 66: halves
    (32, 3, 1984, 704, "2,1,32,1,2", "2,1,32,2,2"),      # 66: halves; 93: halves
    (16, 8, 1280, 640, "2,1,16,1,4", "2,1,32,2,1"),      # 160: quarters; 160: whole
    (16, 8, 1024, 640, "2,1,16,1,4", "2,1,32,2,2"),      # 160; 128: halves
    (16, 2, 1984, 704, "2,1,32,1,2", "1,1,32,2,4"),      # 44 tiles of rows just too narrow for one chain per lane
    (16, 2, 2048, 704, "1,1,32,1,4", "1,1,32,2,4"),
    (256, 8, 128, 704, "2,1,16,1,4", "1,1,32,2,4"),      # as many experts as threads; 176 tiles
    (16, 6, 256, 1024, "4,1,16,1,2", "1,1,32,2,4"),      # 192: four quarters and the publisher would be one too many
    (20, 6, 1920, 1216, "4,1,16,1,2", "2,1,32,2,1"),     # 228: halves with four chains; 180: whole
    (24, 8, 2112, 1344, "4,1,16,1,2", "4,1,16,2,1"),     # 336: halves with four chains; 264: whole with four
    (16, 1, 4160, 64, "1,1,32,1,4", "2,1,32,2,1"),       # counters of halves do not fit: whole tiles
    (300, 3, 1984, 704, "2,1,32,1,2", "2,1,32,2,2"),     # a router of more than 256 experts: no workgroups of 256 threads
    (300, 8, 1280, 640, "2,1,32,1,1", "2,1,32,2,1"),
    (300, 6, 256, 1024, "4,1,16,1,1", "1,1,32,2,4"),     # 192 tiles
    (512, 8, 128, 1024, "4,1,16,1,1", "1,1,32,2,4"),     # 256
    (300, 8, 512, 1152, "4,1,16,1,1", "1,1,32,2,4"),     # 288
    (16, 1, 8256, 128, "2,1,32,1,1", "2,1,32,2,1"),      # too wide a row for parts
])
def test_moe_step_in_parts(pkg, oracle, E, K, H, F, gate_up, down):
    print(f"moe parts E={E} K={K} H={H} F={F}", flush=True)
    pool = synth.expert_pool(E, H, F, 1)
    logits, scale = synth.router_logits(E, 2), np.linspace(0.5, 2.0, E).astype(np.float32)
    layer = pkg.lib.MoeLayer(pool, E, H, F, K)
    for seed in (3, 4, 5):                       # the counters start from zero in every step
        x = synth.activations(H, 1, seed)[0]
        status, sel, w, eo, y = layer.step(logits, scale, x)
        assert pkg.lib.load().salt_mi355_last_kernel().decode() == f"q4_tile_kernel<{gate_up}> + q4_tile_kernel<{down}>"
        osel, ow, oeo, oy = np.zeros(K, np.int32), np.zeros(K, np.float32), np.zeros((K, H), np.float32), np.zeros(H, np.float32)
        assert oracle.orc_moe_decode_step(ct.byref(ExpertGeometry(H, F)), ptr(pool), E, K, ptr(logits), ptr(scale), ptr(x),
                                          ptr(osel), ptr(ow), ptr(oeo), ptr(oy), 2) == 0
        assert status == 0 and np.array_equal(sel, osel) and np.array_equal(bits(w), bits(ow))
        assert np.array_equal(bits(eo), bits(oeo)) and np.array_equal(bits(y), bits(oy))
