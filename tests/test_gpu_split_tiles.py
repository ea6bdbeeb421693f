"""Launches with few tiles, or with up to one and a half per compute unit, run on parts of a tile (sixteen or thirty-two
rows per workgroup, several chain slices per wave): the same bits as the CPU checker at the edges of the parts, of the
tiles, of the rule's ranges and of the columns that the parts keep in LDS."""
import numpy as np
import pytest

from golden import cases
from oracle_lib import bits, host_threads, ptr

pytestmark = pytest.mark.gpu
synth = cases.synth


@pytest.mark.parametrize("R,C", [
    (1, 64), (15, 576), (17, 1088), (63, 2816), (65, 8192), (130, 8256),    # 8256 columns: whole tiles
    (6144, 192), (6145, 192), (8192, 128), (8193, 128),                     # 96, 97, 128 and 129 tiles
])
def test_q4_parts_of_tiles(pkg, oracle, R, C):
    print(f"q4 split R={R} C={C}", flush=True)
    vals, scales, biases = synth.q4_tensor(R, C, R + C)
    if R == 63:
        scales = scales.copy()
        scales[5] = 0x7B80                       # 2^120: the path for scales that the converter's power of two overflows
    x = synth.activations(C, 1, 31)
    got = pkg.lib.q4_matvec(vals, scales, biases, R, C, x)
    want = np.zeros((1, R), np.float32)
    assert oracle.orc_q4_matvec_threads(ptr(vals), ptr(scales), ptr(biases), R, C, ptr(x[0]), ptr(want[0]),
                                        host_threads()) == 0
    assert np.array_equal(bits(got), bits(want))


@pytest.mark.parametrize("R,C,B", [(1, 64, 2), (17, 8256, 3), (65, 576, 4), (6145, 192, 2), (8192, 128, 4), (8193, 128, 3),
                                   (16385, 576, 1), (16500, 512, 2), (20000, 64, 3), (24576, 1088, 4), (24577, 128, 3)])
def test_q4_parts_with_staged_activations(pkg, oracle, R, C, B):
    print(f"q4 staged R={R} C={C} B={B}", flush=True)
    vals, scales, biases = synth.q4_tensor(R, C, R + C)
    xs = synth.activations(C, B, 33)
    got = pkg.lib.q4_matvec(vals, scales, biases, R, C, xs)
    want = np.zeros((B, R), np.float32)
    for t in range(B):
        assert oracle.orc_q4_matvec_threads(ptr(vals), ptr(scales), ptr(biases), R, C, ptr(xs[t]), ptr(want[t]),
                                            host_threads()) == 0
    assert np.array_equal(bits(got), bits(want))


@pytest.mark.parametrize("kernel,rows,C", [
    ("q4_tile_kernel<2,{},16,0,4>", (70, 1, 1040, 333), 576),                     # 24 tiles: quarters
    ("q4_tile_kernel<2,{},16,0,2>", (2112, 2100, 2112, 6), 192),                  # 100 tiles: halves
    ("q4_tile_kernel<4,{},16,0,2>", (2112, 2112, 2100, 2112, 2112, 2111, 2112, 2049), 576),    # 264 tiles: halves, four chains
    ("q4_tile_kernel<4,{},16,0,2>", (8192, 8190, 8130), 128),                     # 384 tiles, the last one of two rows
])
@pytest.mark.parametrize("tokens", [1, 2, 3, 4])
def test_q4_job_tables_in_parts(pkg, oracle, kernel, rows, C, tokens):
    """Several jobs with ragged last tiles, and in the second job a scale that takes the path for scales the converter's power
    of two overflows."""
    if tokens == 1:
        kernel = kernel.replace("<2,{},16", "<2,1,32")
    print(f"q4 jobs in parts {kernel} tokens={tokens}", flush=True)
    lib = pkg.lib.init()
    stream = lib.salt_mi355_stream()
    hold, jobs, want = [], (pkg.lib.Q4Job * len(rows))(), []
    for j, R in enumerate(rows):
        vals, scales, biases = synth.q4_tensor(R, C, 50 + j)
        if j == 1:
            scales = scales.copy()
            scales[-1] = 0x7B80                  # 2^120, in the job's last row
            scales[0] = 0xFB80
        xs = synth.activations(C, tokens, 60 + j)
        y = np.zeros((tokens, R), np.float32)
        for t in range(tokens):
            assert oracle.orc_q4_matvec_threads(ptr(vals), ptr(scales), ptr(biases), R, C, ptr(xs[t]), ptr(y[t]), host_threads()) == 0
        bufs = [pkg.lib.DeviceBuffer.from_host(a) for a in (vals, scales, biases, xs)] + [pkg.lib.DeviceBuffer(y.nbytes, fill=0xFF)]
        jobs[j] = pkg.lib.Q4Job(*[b.ptr for b in bufs], R)
        hold.append(bufs)
        want.append(y)
    pkg.lib.check(lib.salt_mi355_q4_jobs_dev(jobs, len(rows), C, tokens, 0, stream), "q4_jobs_dev")
    pkg.lib.check(lib.salt_mi355_stream_sync(stream), "sync")
    assert lib.salt_mi355_last_kernel().decode() == kernel.format(tokens)
    for bufs, y in zip(hold, want):
        assert np.array_equal(bits(bufs[4].to_host(np.float32).reshape(y.shape)), bits(y))


@pytest.mark.parametrize("R,C", [(1, 64), (31, 544), (33, 4096), (100, 8192), (4096, 96), (4097, 96), (8192, 64), (8193, 64)])
def test_nvfp4_parts_of_tiles(pkg, oracle, R, C):
    print(f"nvfp4 split R={R} C={C}", flush=True)
    packed, scales = synth.nvfp4_tensor(R, C, R + C)
    x = synth.activations(C, 1, 37)[0]
    status, got = pkg.lib.nvfp4_matvec_one_launch(packed, scales, 2688.0, R, C, x)
    want = np.zeros(R, np.float32)
    scratch = (np.zeros(C // 2, np.uint8), np.zeros(C // 16, np.uint8), np.zeros(C, np.float32))
    assert oracle.orc_nvfp4_matvec(ptr(packed), ptr(scales), 2688.0, 64.0, R, C, ptr(x), ptr(want), ptr(scratch[0]),
                                   ptr(scratch[1]), ptr(scratch[2])) == 0
    assert status == 0 and np.array_equal(bits(got), bits(want))
    x[C - 1] = np.nan                            # a rejected activation publishes nothing
    status, got = pkg.lib.nvfp4_matvec_one_launch(packed, scales, 2688.0, R, C, x)
    assert status == -1 and (bits(got) == 0xFFFFFFFF).all()


@pytest.mark.parametrize("E,K,H,F", [(16, 1, 1024, 512), (128, 4, 2816, 704), (300, 2, 512, 576), (512, 1, 256, 64)])
def test_moe_step_gate_up_parts(pkg, oracle, E, K, H, F):
    """Gate and up launches of at most 128 tiles; more than 256 experts take the block-wide router."""
    import ctypes as ct

    from oracle_lib import ExpertGeometry
    print(f"moe split E={E} K={K} H={H} F={F}", flush=True)
    pool = synth.expert_pool(E, H, F, 1)
    logits, scale, x = synth.router_logits(E, 2), np.linspace(0.5, 2.0, E).astype(np.float32), synth.activations(H, 1, 3)[0]
    status, sel, w, eo, y = pkg.lib.MoeLayer(pool, E, H, F, K).step(logits, scale, x)
    osel, ow, oeo, oy = np.zeros(K, np.int32), np.zeros(K, np.float32), np.zeros((K, H), np.float32), np.zeros(H, np.float32)
    assert oracle.orc_moe_decode_step(ct.byref(ExpertGeometry(H, F)), ptr(pool), E, K, ptr(logits), ptr(scale), ptr(x),
                                      ptr(osel), ptr(ow), ptr(oeo), ptr(oy), 2) == 0
    assert status == 0 and np.array_equal(sel, osel) and np.array_equal(bits(w), bits(ow))
    assert np.array_equal(bits(eo), bits(oeo)) and np.array_equal(bits(y), bits(oy))
