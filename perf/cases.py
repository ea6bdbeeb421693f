"""The work that users of this backend have it do, as cases that a timing harness can prepare, run and compare.

A case is a dict of plain values; `kind` names the entry point:

  q4            affine-Q4 decode matvecs (salt_mi355_q4_matvec_dev / _jobs_dev; cls "t": the tolerance-class forms)
  nvfp4         NVFP4 reference matvecs including the activation pass (cls as above)
  q4_matmul     prefill-sized affine-Q4 matmul          nvfp4_matmul  prefill-sized NVFP4 matmul
  moe_decode    one token through one MoE layer         moe_prefill   many tokens through one MoE layer
  ffn_block     the feed-forward half of a decoder layer for one token
  head          bf16 language-model head
  abi_chain     the engine ABI's decode call for routed experts, host pointers in and out
  abi_matvec    the engine ABI's single projection, host pointers in and out

Device-resident kinds run on the library's own stream and return the buffers that they wrote.
"""
import ctypes as C
import itertools
import math

import numpy as np
import torch

from __graft_entry__ import load_package

gpu = load_package().lib
GROUP = 64
DIVISOR, INPUT_SCALE = 2688.0, 64.0     # NVFP4 per-tensor factors, as the benchmark and the tests use them


# ------------------------------------------------------------------------------------------------ the cases

def listed():
    return [
        # One attention-output-sized projection of a decode step on the default (bit-exact) class: the smallest launch.
        {"name": "q4_one_2816", "kind": "q4", "cls": "exact", "R": 2816, "C": 2816, "B": 1, "mats": 1},
        # Dense gate/up projections of four layers for a batch of three sequences, bit-exact, rows no multiple of a tile.
        {"name": "q4_batch3", "kind": "q4", "cls": "exact", "R": 2112, "C": 2816, "B": 3, "mats": 8},
        # The decode sweep's widest shape, many matrices in one launch, tolerance class: the bandwidth-bound form.
        {"name": "q4_t_sweep", "kind": "q4", "cls": "t", "R": 16384, "C": 2816, "B": 1, "mats": 24},
        # The NVFP4 matvec of one token, bit-exact, one matrix per launch.
        {"name": "nvfp4_one_8192", "kind": "nvfp4", "cls": "exact", "R": 8192, "C": 8192, "B": 1, "mats": 1},
        # Several NVFP4 matrices in one launch, tolerance class.
        {"name": "nvfp4_t_x6", "kind": "nvfp4", "cls": "t", "R": 8192, "C": 8192, "B": 1, "mats": 6},
        # A 256-token prompt against one NVFP4 matrix.
        {"name": "nvfp4_matmul_256", "kind": "nvfp4_matmul", "R": 8192, "C": 8192, "B": 256},
        # A prompt of 333 tokens against one wide Q4 projection.
        {"name": "q4_matmul_333", "kind": "q4_matmul", "R": 16384, "C": 2816, "B": 333},
        # One token through one routed layer (E = 128, top-8), tolerance class.
        {"name": "moe_decode_t", "kind": "moe_decode", "cls": "t", "E": 128, "K": 8, "H": 2816, "F": 704},
        # A prompt of 2048 tokens through the same layer, popularity of experts ~ 1/rank^1.1.
        {"name": "moe_prefill_2048", "kind": "moe_prefill", "E": 128, "K": 8, "H": 2816, "F": 704, "T": 2048},
        # The whole feed-forward half of a decoder layer (norms, dense branch, router gate, experts, combine), bit-exact.
        {"name": "ffn_block", "kind": "ffn_block", "E": 128, "K": 8, "H": 2816, "D": 2112, "F": 704},
        # The language-model head of one token.
        {"name": "head_262144", "kind": "head", "R": 262144, "C": 2816, "B": 1},
        # The engine's own decode call over eight selected experts, host pointers, synchronous.
        {"name": "abi_chain_8", "kind": "abi_chain", "E": 24, "K": 8, "H": 2816, "F": 704},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cols(rng, lo, hi):
    return max(GROUP, _log(rng, lo, hi) // GROUP * GROUP)


def draw(rng):
    kind = rng.choice(["q4", "q4", "q4", "nvfp4", "nvfp4", "nvfp4_matmul", "q4_matmul", "moe_decode", "moe_decode",
                       "moe_prefill", "ffn_block", "head", "abi_chain", "abi_matvec"])
    if kind in ("q4", "nvfp4"):
        case = {"kind": kind, "cls": rng.choice(["exact", "t"]), "R": _log(rng, 256, 16384), "C": _cols(rng, 512, 8192),
                "B": rng.choice([1, 1, 1, 2, 3, 4]) if kind == "q4" else 1}
        most = max(1, int(600e6 / (0.5625 * case["R"] * case["C"] * case["B"])))
        case["mats"] = 1 if rng.random() < 0.4 else min(most, rng.randint(2, 24))
        return case
    if kind in ("q4_matmul", "nvfp4_matmul"):
        case = {"kind": kind, "R": _log(rng, 512, 16384), "C": _cols(rng, 512, 8192), "B": _log(rng, 33, 1024)}
        while 2.0 * case["R"] * case["C"] * case["B"] > 6e10:
            case["B"] = max(33, case["B"] // 2)
            case["R"] = max(512, case["R"] * 3 // 4)
        return case
    if kind == "head":
        return {"kind": kind, "R": _log(rng, 32000, 262144), "C": _cols(rng, 1024, 2816), "B": rng.choice([1, 1, 2])}
    if kind == "abi_matvec":
        return {"kind": kind, "R": _log(rng, 512, 8192), "C": _cols(rng, 512, 8192)}
    case = {"kind": kind, "E": rng.choice([16, 32, 60, 64, 128]), "K": rng.choice([1, 2, 4, 6, 8]),
            "H": _cols(rng, 1024, 2816), "F": _cols(rng, 512, 1024)}
    if kind == "moe_decode":
        case["cls"] = rng.choice(["exact", "t"])
    elif kind == "moe_prefill":
        case["T"] = _log(rng, 64, 2048)
    elif kind == "ffn_block":
        case["D"] = _cols(rng, 1024, 2816)
    else:
        case["E"] = rng.choice([8, 16, 24])
    return case


def _proj_bytes(H, F):
    return H * F // 2 + 4 * (H * F // GROUP)


def work(case):
    kind = case["kind"]
    if kind in ("q4", "nvfp4"):
        R, Cc, B, n = case["R"], case["C"], case["B"], case["mats"]
        return {"bytes": n * (0.5625 * R * Cc + 4.0 * B * R) + 4.0 * B * Cc, "flops": 2.0 * n * R * Cc * B}
    if kind in ("q4_matmul", "nvfp4_matmul"):
        R, Cc, B = case["R"], case["C"], case["B"]
        return {"bytes": 0.5625 * R * Cc + 4.0 * B * (R + Cc), "flops": 2.0 * R * Cc * B}
    if kind == "head":
        R, Cc, B = case["R"], case["C"], case["B"]
        return {"bytes": 2.0 * R * Cc + 4.0 * B * (R + Cc), "flops": 2.0 * R * Cc * B}
    if kind == "abi_matvec":
        R, Cc = case["R"], case["C"]
        return {"bytes": 0.5625 * R * Cc + 4.0 * (R + Cc), "flops": 2.0 * R * Cc}
    H, F, K = case["H"], case["F"], case["K"]
    experts, rows = K, K
    if kind == "moe_prefill":
        experts, rows = min(case["E"], K * case["T"]), K * case["T"]
    tokens = case.get("T", 1)
    total = experts * 3.0 * _proj_bytes(H, F) + 8.0 * tokens * H
    flops = 6.0 * rows * H * F
    if kind == "abi_chain":
        total = K * (3.0 * _proj_bytes(H, F) + 8.0 * H)
    if kind == "ffn_block":
        total += 3.0 * _proj_bytes(H, case["D"]) + case["E"] * H * (1 + 4 / GROUP) + 28.0 * H
        flops += 6.0 * H * case["D"] + 2.0 * H * case["E"]
    return {"bytes": total, "flops": flops}


def tolerance(case):
    """Bit-exact entry points publish the reference CPU kernels' bits.  The others: four times the measured distance
    from the same products and sums in 64 bits."""
    kind = case["kind"]
    if kind in ("ffn_block", "head", "abi_chain", "abi_matvec") or case.get("cls") == "exact":
        return "exact"
    return {"rel": {"q4": 6e-7, "nvfp4": 8e-7, "nvfp4_matmul": 5e-7, "moe_decode": 1.1e-6, "q4_matmul": 4e-6,
                    "moe_prefill": 8e-6}[kind]}


# ------------------------------------------------------------------------------------------------ inputs

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _bytes(g, *shape):
    return torch.randint(0, 256, shape, generator=g, device="cuda", dtype=torch.uint8)


def _uniform(g, lo, hi, *shape):
    return torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo


def _normal(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _raw(t):
    return t.contiguous().view(torch.uint8)


def _q4_blobs(g, count, n):
    """[count][values | scales | biases] of n-element affine-Q4 matrices: uniform codes, scales in [0.005, 0.02], biases
    that centre a group on zero give or take 1e-3."""
    groups = n // GROUP
    blob = _bytes(g, count, n // 2 + 4 * groups)
    scales = _uniform(g, 0.005, 0.02, count, groups).bfloat16()
    biases = (-8.0 * scales.float() + 1e-3 * _normal(g, count, groups)).bfloat16()
    blob[:, n // 2:n // 2 + 2 * groups] = _raw(scales).view(count, 2 * groups)
    blob[:, n // 2 + 2 * groups:] = _raw(biases).view(count, 2 * groups)
    return blob


def _q4_parts(address, n):
    return address, address + n // 2, address + n // 2 + 2 * (n // GROUP)


def _pool(g, E, H, F):
    return _q4_blobs(g, E * 3, H * F).view(E, 3 * _proj_bytes(H, F))


def _nvfp4(g, count, R, Cc):
    """Packed E2M1 codes [count][R][C/2] and E4M3 block scales between 2^-6 and 2^4."""
    return _bytes(g, count, R, Cc // 2), torch.randint(0x08, 0x59, (count, R, Cc // 16), generator=g, device="cuda",
                                                       dtype=torch.uint8)


def _empty(*shape, dtype=torch.float32):
    return torch.zeros(shape, device="cuda", dtype=dtype)


class State:
    """The call a user's program repeats: `call()` enqueues it, `outputs` are the buffers that it writes."""

    def __init__(self, fn, args, outputs, keep, close=None):
        self.fn, self.args, self.outputs, self.keep, self.close = fn, args, outputs, keep, close

    def __del__(self):
        if self.close is not None:
            self.close()


def _q4_state(case, g, lib, stream):
    R, Cc, B, n = case["R"], case["C"], case["B"], case["mats"]
    w, xs, ys = _q4_blobs(g, n, R * Cc), _normal(g, B, Cc), _empty(n, B, R)
    parts = [_q4_parts(w[j].data_ptr(), R * Cc) for j in range(n)]
    if n == 1:
        args = [*parts[0], R, Cc, B, xs.data_ptr(), ys.data_ptr()]
        if case["cls"] == "t":
            return State(lib.salt_mi355_q4_matvec_t_dev, (*args, stream), ys, (w, xs))
        return State(lib.salt_mi355_q4_matvec_dev, (*args, 0, stream), ys, (w, xs))
    jobs = (gpu.Q4Job * n)(*[gpu.Q4Job(*parts[j], xs.data_ptr(), ys[j].data_ptr(), R) for j in range(n)])
    if case["cls"] == "t":
        return State(lib.salt_mi355_q4_jobs_t_dev, (jobs, n, Cc, B, stream), ys, (w, xs))
    return State(lib.salt_mi355_q4_jobs_dev, (jobs, n, Cc, B, 0, stream), ys, (w, xs))


def _nvfp4_state(case, g, lib, stream):
    R, Cc, n = case["R"], case["C"], case["mats"]
    (w, s), xs, ys, status = _nvfp4(g, n, R, Cc), _normal(g, 1, Cc), _empty(n, 1, R), _empty(1, dtype=torch.int32)
    if n == 1:
        head = [w.data_ptr(), s.data_ptr(), DIVISOR, INPUT_SCALE, R, Cc]
        tail = [xs.data_ptr(), ys.data_ptr(), status.data_ptr()]
        if case["cls"] == "t":
            return State(lib.salt_mi355_nvfp4_matvec_t_dev, (*head, 1, *tail, stream), [ys, status], (w, s, xs))
        return State(lib.salt_mi355_nvfp4_matvec_qdq_dev, (*head, *tail, 0, stream), [ys, status], (w, s, xs))
    dq = _empty(1, Cc)
    source = xs if case["cls"] == "t" else dq
    jobs = (gpu.Fp4Job * n)(*[gpu.Fp4Job(w[j].data_ptr(), s[j].data_ptr(), DIVISOR, source.data_ptr(), ys[j].data_ptr(), R)
                              for j in range(n)])
    if case["cls"] == "t":
        return State(lib.salt_mi355_nvfp4_jobs_t_dev, (jobs, n, Cc, 1, INPUT_SCALE, status.data_ptr(), stream), [ys, status],
                     (w, s, xs))

    def both():
        rc = lib.salt_mi355_nvfp4_qdq_dev(xs.data_ptr(), Cc, 1, INPUT_SCALE, None, None, dq.data_ptr(), status.data_ptr(),
                                          stream)
        return rc or lib.salt_mi355_nvfp4_jobs_dev(jobs, n, Cc, 1, 0, stream)
    return State(both, (), [ys, status], (w, s, xs, dq))


def _q4_matmul_state(case, g, lib, stream):
    R, Cc, B = case["R"], case["C"], case["B"]
    w, xs, ys = _q4_blobs(g, 1, R * Cc), _normal(g, B, Cc), _empty(B, R)
    ws = _empty(lib.salt_mi355_q4_matmul_workspace_bytes(Cc, B), dtype=torch.uint8)
    args = (*_q4_parts(w.data_ptr(), R * Cc), R, Cc, B, xs.data_ptr(), ys.data_ptr(), ws.data_ptr(), stream)
    return State(lib.salt_mi355_q4_matmul_dev, args, ys, (w, xs, ws))


def _nvfp4_matmul_state(case, g, lib, stream):
    R, Cc, B = case["R"], case["C"], case["B"]
    (w, s), xs, ys, status = _nvfp4(g, 1, R, Cc), _normal(g, B, Cc), _empty(B, R), _empty(1, dtype=torch.int32)
    ws = _empty(lib.salt_mi355_nvfp4_matmul_workspace_bytes(R, Cc, B), dtype=torch.uint8)
    args = (w.data_ptr(), s.data_ptr(), DIVISOR, INPUT_SCALE, R, Cc, B, xs.data_ptr(), ys.data_ptr(), status.data_ptr(),
            ws.data_ptr(), stream)
    return State(lib.salt_mi355_nvfp4_matmul_dev, args, [ys, status], (w, s, xs, ws))


def _moe_decode_state(case, g, lib, stream):
    E, K, H, F = case["E"], case["K"], case["H"], case["F"]
    pool, logits, scale, x = _pool(g, E, H, F), _normal(g, E), _uniform(g, 0.5, 2.0, E), _normal(g, H)
    sel, wts, eo, out = _empty(K, dtype=torch.int32), _empty(K), _empty(K, H), _empty(H)
    ws = _empty(lib.salt_mi355_moe_workspace_bytes(H, F, E, K), dtype=torch.uint8)
    fn = lib.salt_mi355_moe_decode_step_t_dev if case["cls"] == "t" else lib.salt_mi355_moe_decode_step_dev
    args = (pool.data_ptr(), pool.shape[1], H, F, E, K, *[t.data_ptr() for t in (logits, scale, x, sel, wts, eo, out, ws)],
            stream)
    return State(fn, args, [sel, wts, eo, out], (pool, logits, scale, x, ws))


def _moe_prefill_state(case, g, lib, stream):
    E, K, H, F, T = case["E"], case["K"], case["H"], case["F"], case["T"]
    pool, xs, out = _pool(g, E, H, F), _normal(g, T, H), _empty(T, H)
    # K distinct experts per token, popularity ~ 1/rank^1.1 (Gumbel top-k), ids ascending, weights a softmax
    rank = torch.randperm(E, generator=g, device="cuda") + 1
    keys = -1.1 * torch.log(rank.float()) - torch.log(-torch.log(_uniform(g, 1e-7, 1 - 1e-7, T, E)))
    sel = keys.topk(K, dim=1).indices.sort(dim=1).values.int().contiguous()
    wts = torch.softmax(_normal(g, T, K), dim=1).contiguous()
    rows, pairs, status = _empty(E, dtype=torch.int32), _empty(T * K, dtype=torch.int32), _empty(1, dtype=torch.int32)
    ws = _empty(lib.salt_mi355_moe_prefill_workspace_bytes(H, F, E, K, T), dtype=torch.uint8)
    args = (pool.data_ptr(), pool.shape[1], H, F, E, K, T,
            *[t.data_ptr() for t in (sel, wts, xs, out, rows, pairs, status, ws)], stream)
    return State(lib.salt_mi355_moe_prefill_dev, args, [out, rows, pairs, status], (pool, sel, wts, xs, ws))


def _ffn_state(case, g, lib, stream):
    E, K, H, D, F = case["E"], case["K"], case["H"], case["D"], case["F"]
    desc = gpu.FfnLayerDesc(H, D, F, E, K, 1e-6, 0.61)
    keep = []

    def put(t):
        keep.append(t)
        return t.data_ptr()

    for name in ("pre_norm", "pre_norm_2", "post_norm_1", "post_norm_2", "post_norm"):
        setattr(desc, name, put(1.0 + 0.1 * _normal(g, H)))
    desc.router_scale = put(1.0 + 0.3 * _normal(g, H))
    desc.per_expert_scale = put(_uniform(g, 0.5, 2.0, E))
    for name in ("dense_gate", "dense_up", "dense_down"):
        setattr(desc, name, (C.c_void_p * 3)(*_q4_parts(put(_q4_blobs(g, 1, H * D)), H * D)))
    groups = -(-E * H // GROUP)
    desc.router = (C.c_void_p * 3)(put(_bytes(g, E * H)), put(_uniform(g, 0.0003, 0.0006, groups).bfloat16()),
                                   put(_uniform(g, -0.07, -0.04, groups).bfloat16()))
    pool = _pool(g, E, H, F)
    desc.pool, desc.expert_stride = put(pool), pool.shape[1]
    residual, out = 3.0 * _normal(g, H), _empty(H)
    sel, wts, status = _empty(K, dtype=torch.int32), _empty(K), _empty(1, dtype=torch.int32)
    ws = _empty(lib.salt_mi355_ffn_block_workspace_bytes(C.byref(desc)), dtype=torch.uint8)
    args = (C.byref(desc), *[t.data_ptr() for t in (residual, out, sel, wts, status, ws)], stream)
    return State(lib.salt_mi355_ffn_block_dev, args, [out, sel, wts, status], (desc, keep, residual, ws))


def _head_state(case, g, lib, stream):
    R, Cc, B = case["R"], case["C"], case["B"]
    w, xs, ys = (0.02 * _normal(g, R, Cc)).bfloat16(), _normal(g, B, Cc), _empty(B, R)
    return State(lib.salt_mi355_bf16_matvec_dev, (w.data_ptr(), R, Cc, B, xs.data_ptr(), None, ys.data_ptr(), stream), ys,
                 (w, xs))


class _Expert(C.Structure):             # SaltGpuMoeExpert of include/salt_gpu_mi355_engine.h
    _fields_ = [(p + f, C.c_void_p) for p in ("gate", "up", "down") for f in ("_vals", "_scales", "_biases", "_id")] + [
        ("group", C.c_int), ("resource_slot", C.c_int), ("logical_resource_id", C.c_uint64)]


_resource = itertools.count(5000)


def _host(t):
    return t.cpu().numpy()


def _engine(lib):
    vp, i, u, sz = C.c_void_p, C.c_int, C.c_uint32, C.c_size_t
    for name, args in (("salt_gpu_init", ()), ("salt_gpu_weight_resource_describe", (u, u, vp, sz)),
                       ("salt_gpu_weight_resource_activate", (u, u, i)), ("salt_gpu_weight_resource_deactivate", (u, u)),
                       ("salt_gpu_q4_matvec", (vp, vp, vp, i, i, vp, vp)),
                       ("salt_gpu_expert_resource_bind", (u, vp, sz)), ("salt_gpu_expert_resource_unbind", (u,)),
                       ("salt_gpu_q4_moe_chain", (vp, i, i, i, vp, vp, vp, vp, sz))):
        fn = getattr(lib, name)
        fn.restype, fn.argtypes = i, list(args)
    gpu.check(lib.salt_gpu_init(), "salt_gpu_init")
    return next(_resource)


def _abi_chain_state(case, g, lib, stream):
    E, K, H, F = case["E"], case["K"], case["H"], case["F"]
    rid = _engine(lib)
    pool, proj = _host(_pool(g, E, H, F)), _proj_bytes(H, F)
    chosen = sorted(torch.randperm(E, generator=g, device="cuda")[:K].tolist())
    gpu.check(lib.salt_gpu_expert_resource_bind(rid, pool.ctypes.data, pool.nbytes), "expert_resource_bind")
    records = (_Expert * K)()
    for record, e in zip(records, chosen):
        for p, name in enumerate(("gate", "up", "down")):
            v, s, b = _q4_parts(pool.ctypes.data + (e * 3 + p) * proj, H * F)
            for field, value in (("_vals", v), ("_scales", s), ("_biases", b), ("_id", v)):
                setattr(record, name + field, value)
        record.group, record.resource_slot, record.logical_resource_id = 1, -1, 0
    x = np.tile(_host(_normal(g, H)), (K, 1))
    y, scratch = np.zeros((K, H), np.float32), np.zeros((2, K * F), np.float32)
    args = (C.addressof(records), K, H, F, x.ctypes.data, y.ctypes.data, scratch[0].ctypes.data, scratch[1].ctypes.data, K * F)
    return State(lib.salt_gpu_q4_moe_chain, args, y, (pool, records, x, scratch),
                 lambda: lib.salt_gpu_expert_resource_unbind(rid))


def _abi_matvec_state(case, g, lib, stream):
    R, Cc = case["R"], case["C"]
    rid = _engine(lib)
    blob, x, y = _host(_q4_blobs(g, 1, R * Cc)), _host(_normal(g, Cc)), np.zeros(R, np.float32)
    gpu.check(lib.salt_gpu_weight_resource_describe(1, rid, blob.ctypes.data, blob.nbytes), "weight_resource_describe")
    gpu.check(lib.salt_gpu_weight_resource_activate(1, rid, 2), "weight_resource_activate")
    args = (*_q4_parts(blob.ctypes.data, R * Cc), R, Cc, x.ctypes.data, y.ctypes.data)
    return State(lib.salt_gpu_q4_matvec, args, y, (blob, x), lambda: lib.salt_gpu_weight_resource_deactivate(1, rid))


_STATES = {"q4": _q4_state, "nvfp4": _nvfp4_state, "q4_matmul": _q4_matmul_state, "nvfp4_matmul": _nvfp4_matmul_state,
           "moe_decode": _moe_decode_state, "moe_prefill": _moe_prefill_state, "ffn_block": _ffn_state, "head": _head_state,
           "abi_chain": _abi_chain_state, "abi_matvec": _abi_matvec_state}


def prepare(case, seed):
    lib = gpu.init()
    state = _STATES[case["kind"]](case, _generator(seed), lib, lib.salt_mi355_stream())
    torch.cuda.synchronize()
    return state


def run(state):
    gpu.check(state.fn(*state.args), "call")
    return state.outputs


# ------------------------------------------------------------------------------------------------ the same in 64 bits

def _q4_rows(blob, R, Cc):
    """One matrix of _q4_blobs as float64 [R][Cc]."""
    n = R * Cc
    v = blob[:n // 2]
    q = torch.stack((v & 15, v >> 4), 1).view(R, Cc // GROUP, GROUP).double()
    s, b = (blob[n // 2 + 2 * k * (n // GROUP):][:2 * (n // GROUP)].clone().view(torch.bfloat16).double().view(R, -1, 1)
            for k in (0, 1))
    return q.mul_(s).add_(b).view(R, Cc)


def _q4_product(blob, R, Cc, xs):
    """xs [B][Cc] (float64) times the matrix, in slabs of rows."""
    n, slab, outs = R * Cc, 4096, []
    groups = Cc // GROUP
    for r in range(0, R, slab):
        m = min(slab, R - r)
        part = torch.cat((blob[r * Cc // 2:(r + m) * Cc // 2], blob[n // 2 + 2 * r * groups:n // 2 + 2 * (r + m) * groups],
                          blob[n // 2 + 2 * (R + r) * groups:n // 2 + 2 * (R + r + m) * groups]))
        outs.append(xs @ _q4_rows(part, m, Cc).T.contiguous())
    return torch.cat(outs, 1)


def _e2m1(codes):
    table = torch.tensor([0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0], device="cuda", dtype=torch.float64)
    mag = table[(codes & 7).long()]
    return torch.where(codes > 7, -mag, mag)


def _fp4_values(w, s):
    R, half = w.shape
    v = torch.stack((w & 15, w >> 4), 2).view(R, half // 8, 16)
    return (_e2m1(v) * s.view(torch.float8_e4m3fn).double().unsqueeze(2)).view(R, 2 * half) / DIVISOR


def _fp4_activations(xs):
    """The NVFP4 image of the activations: which code an element gets is decided in 32 bits, as the format's quantiser does."""
    v = xs.view(xs.shape[0], -1, 16)
    raw = (INPUT_SCALE * (v.abs().amax(2, keepdim=True) * torch.tensor(1 / 6, device="cuda"))).clamp(max=448.0)
    scale = raw.to(torch.float8_e4m3fn).float()
    to_code = torch.where(scale == 0, torch.zeros_like(scale), INPUT_SCALE / scale)
    m = (v * to_code).clamp(-6.0, 6.0)
    a = m.abs()
    code = sum((test.to(torch.uint8) for test in (a > 0.25, a >= 0.75, a > 1.25, a >= 1.75, a > 2.5, a >= 3.5, a > 5.0)))
    return (_e2m1(code) * torch.sign(m).double() * (scale / INPUT_SCALE).double()).view(xs.shape)


def _fp4_product(w, s, xs, slab=2048):
    return torch.cat([xs @ _fp4_values(w[r:r + slab], s[r:r + slab]).T.contiguous() for r in range(0, w.shape[0], slab)], 1)


def _gelu(v):
    return 0.5 * v * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (v + 0.044715 * v ** 3)))


def _expert(blobs, H, F, xs):
    """Output of the expert with the three matrices blobs for the rows xs (float64)."""
    gate, up, down = blobs.view(3, -1)
    return _q4_product(down, H, F, _gelu(_q4_product(gate, F, H, xs)) * _q4_product(up, F, H, xs))


def exact(case, seed):
    kind, g = case["kind"], _generator(seed)
    status = torch.zeros(1, device="cuda", dtype=torch.int32)
    if kind in ("q4", "q4_matmul"):
        R, Cc, B, n = case["R"], case["C"], case["B"], case.get("mats", 1)
        w, xs = _q4_blobs(g, n, R * Cc), _normal(g, B, Cc).double()
        ys = torch.stack([_q4_product(w[j], R, Cc, xs) for j in range(n)])
        return ys if kind == "q4" else ys[0]
    if kind in ("nvfp4", "nvfp4_matmul"):
        R, Cc, B, n = case["R"], case["C"], case.get("B", 1), case.get("mats", 1)
        (w, s), xs = _nvfp4(g, n, R, Cc), _normal(g, B, Cc)
        xs = _fp4_activations(xs)
        ys = torch.stack([_fp4_product(w[j], s[j], xs) for j in range(n)])
        return [ys if kind == "nvfp4" else ys[0], status]
    if kind == "head":
        R, Cc, B = case["R"], case["C"], case["B"]
        w, xs = (0.02 * _normal(g, R, Cc)).bfloat16(), _normal(g, B, Cc).double()
        return torch.cat([xs @ w[r:r + 16384].double().T.contiguous() for r in range(0, R, 16384)], 1)
    if kind == "abi_matvec":
        R, Cc = case["R"], case["C"]
        blob, x = _q4_blobs(g, 1, R * Cc), _normal(g, Cc).double()
        return _host(_q4_product(blob[0], R, Cc, x[None])[0])
    if kind == "ffn_block":             # a router's choice between near-equal gates is not a number to compare
        return None
    E, K, H, F = case["E"], case["K"], case["H"], case["F"]
    pool = _pool(g, E, H, F)
    if kind == "abi_chain":
        chosen = sorted(torch.randperm(E, generator=g, device="cuda")[:K].tolist())
        x = _normal(g, H).double()[None]
        return _host(torch.cat([_expert(pool[e], H, F, x) for e in chosen]))
    if kind == "moe_decode":
        logits, scale, x = _normal(g, E), _uniform(g, 0.5, 2.0, E), _normal(g, H).double()[None]
        sel = logits.topk(K).indices.sort().values
        wts = torch.softmax(logits[sel].double(), 0) * scale[sel].double()
        eo = torch.cat([_expert(pool[e], H, F, x) for e in sel.tolist()])
        return [sel.int(), wts, eo, wts @ eo]
    T = case["T"]
    xs = _normal(g, T, H).double()
    rank = torch.randperm(E, generator=g, device="cuda") + 1
    keys = -1.1 * torch.log(rank.float()) - torch.log(-torch.log(_uniform(g, 1e-7, 1 - 1e-7, T, E)))
    sel = keys.topk(K, dim=1).indices.sort(dim=1).values
    wts = torch.softmax(_normal(g, T, K), dim=1).double()
    out = torch.zeros(T, H, device="cuda", dtype=torch.float64)
    for e in range(E):
        token, k = (sel == e).nonzero(as_tuple=True)
        if token.numel():
            out.index_add_(0, token, _expert(pool[e], H, F, xs[token]) * wts[token, k][:, None])
    return [out, torch.bincount(sel.flatten(), minlength=E).int(), sel.flatten().argsort(stable=True).int(), status]
