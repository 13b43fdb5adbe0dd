"""Timed cases: what programs ask of the library, through the Python mirror of the HCCL C API.

All ranks of a communicator are driven from one thread on one stream, and a program keeps its communicators, so those are
made once per process and settings.  Buffers, and for the all-to-all-v the count tables, belong to a state.  Results are
defined bit for bit by the schedule (association, operand order, rounding after every step), so every case compares exactly.
"""
import importlib.util
import math
import os
import statistics
import sys

import numpy as np
import torch

_NAME = "cann_hccl_amd_perf"


def _package():
    """The package of the working folder.  Its directory's name holds a hyphen: it is loaded from its path."""
    if _NAME not in sys.modules:
        spec = importlib.util.spec_from_file_location(_NAME, os.path.join(os.getcwd(), "cann-hccl_amd", "__init__.py"))
        mod = importlib.util.module_from_spec(spec)
        sys.modules[_NAME] = mod
        spec.loader.exec_module(mod)
    return sys.modules[_NAME]


_UNIT = {"fp32": 4, "fp16": 2, "bf16": 2, "int8": 1, "int32": 4, "int64": 8}
_TORCH = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16, "int8": torch.int8, "int32": torch.int32, "int64": torch.int64}
_OP = {"sum": 0, "prod": 1, "max": 2, "min": 3}


def _case(name, coll, ranks, count, dtype, algo="ring", op="sum", servers=1, in_place=False, shift=0):
    """`count` elements: the whole buffer of a rank (all-reduce), the received block (reduce-scatter), the sent
    block (all-gather), the median block per pair of ranks (all-to-all-v).  `shift`: elements by which every buffer starts
    behind a 512-byte boundary (a view into a larger allocation)."""
    return {"name": name, "coll": coll, "ranks": ranks, "count": count, "dtype": dtype, "algo": algo, "op": op, "servers": servers,
            "in_place": in_place, "shift": shift}


def listed():
    return [
        # a few numbers everybody needs: loss, gradient norm, overflow flags; the bottom of the benchmark's size sweep
        _case("allreduce_8k", "all_reduce", 8, 2048, "fp32"),
        # one decoding step's activations (64 tokens x 8192) between the ranks of a tensor-parallel layer
        _case("allreduce_bf16_1m", "all_reduce", 8, 64 * 8192, "bf16"),
        # a bucket of gradients, reduced where it lies inside a flat buffer: odd length, odd start.  max, as it may be repeated
        _case("allreduce_bucket_ragged", "all_reduce", 8, 13_107_203, "fp16", op="max", in_place=True, shift=3),
        # the headline: 8 ranks x 256 MiB fp32 sum
        _case("allreduce_256m", "all_reduce", 8, 64 << 20, "fp32"),
        # two servers of four devices: mesh inside, halving-doubling between
        _case("allreduce_two_level_64m", "all_reduce", 8, 16 << 20, "fp32", algo="auto", servers=2),
        # halving-doubling over 32 ranks x 128 MiB of bf16
        _case("allreduce_rhd_32x128m", "all_reduce", 32, 64 << 20, "bf16", algo="rhd"),
        # gradients of a sharded optimizer, 64 MiB per rank in
        _case("reduce_scatter_64m", "reduce_scatter", 8, 4 << 20, "bf16"),
        # the same for quantised values with blocks of odd length, which start at any byte of the send buffers
        _case("reduce_scatter_int8_ragged", "reduce_scatter", 8, 3_000_017, "int8"),
        # parameters of a sharded layer gathered into buffers of which every rank holds its own block already
        _case("allgather_in_place_ragged", "all_gather", 8, 2_621_447, "bf16", in_place=True),
        # the large all-gather of the benchmark: 32 MiB per rank in, 256 MiB out
        _case("allgather_32m", "all_gather", 8, 8 << 20, "fp32"),
        # tokens to experts and back, 16 ranks, lognormal blocks (median 64 Ki elements)
        _case("alltoallv_16", "all_to_all_v", 16, 65536, "int32"),
        # the same in decoding: 64 ranks, blocks of a few hundred bytes
        _case("alltoallv_64_short", "all_to_all_v", 64, 64, "int32"),
    ]


def _log(rng, lo, hi):
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return n if rng.random() < 0.5 else max(lo, n // 64 * 64)


def draw(rng):
    coll = rng.choice(["all_reduce", "all_reduce", "all_reduce", "reduce_scatter", "reduce_scatter", "all_gather", "all_gather", "all_to_all_v"])
    dtype = rng.choice(["fp32", "bf16", "bf16", "fp16", "int8", "int32", "int64"])
    unit = _UNIT[dtype]
    shift = rng.choice([0, 0, 0, 1, 3, 8])
    if coll == "all_to_all_v":
        ranks = rng.choice([8, 16, 16, 32, 64])
        return _unnamed(coll, ranks, _log(rng, 32, (256 << 20) // (ranks * ranks * unit)), dtype)
    algo = rng.choice(["ring", "ring", "mesh", "rhd"])
    servers, in_place, op = 1, False, "sum"
    if coll == "all_reduce":
        ranks = rng.choice([2, 4, 8, 8, 8, 16, 24, 32])
        if algo == "rhd" and ranks == 8 and rng.random() < 0.5:
            algo, servers = "auto", 2
        in_place = rng.random() < 0.3
        op = "max" if in_place else rng.choice(["sum", "sum", "max", "min"])
        # 2 KiB ... 256 MiB per rank, at most 4 GiB on either side
        count = _log(rng, 2048 // unit, min(256 << 20, (4 << 30) // ranks) // unit)
    elif coll == "reduce_scatter":
        ranks = rng.choice([2, 4, 8, 8, 8, 16])
        op = rng.choice(["sum", "sum", "sum", "prod", "max", "min"])
        count = _log(rng, 512 // unit, (1 << 30) // (ranks * ranks) // unit)
    else:
        ranks = rng.choice([2, 4, 8, 8, 8, 16])
        in_place = rng.random() < 0.4
        count = _log(rng, 512 // unit, (2 << 30) // (ranks * ranks) // unit)
    return _unnamed(coll, ranks, count, dtype, algo, op, servers, in_place, shift)


def _unnamed(*args):
    c = _case("", *args)
    del c["name"]
    return c


_communicators = {}


def _communicator(case):
    key = (case["ranks"], case["algo"], case["servers"])
    if key not in _communicators:
        H = _package()
        comms = H.comm_init_all(case["ranks"])
        H.set_param(comms[0], "algo", case["algo"])
        H.set_param(comms[0], "servers", case["servers"])
        _communicators[key] = (comms, torch.cuda.Stream())
    return _communicators[key]


def _fill(t, gen):
    """Normal values; integers over their full range, 64-bit ones within 2^40."""
    if t.is_floating_point():
        t.normal_(generator=gen)
    elif t.dtype == torch.int64:
        t.random_(-(1 << 40), 1 << 40, generator=gen)
    else:
        info = torch.iinfo(t.dtype)
        t.random_(info.min, info.max + 1, generator=gen)


def _buffer(case, n, gen=None):
    whole = torch.zeros(n + case["shift"], dtype=_TORCH[case["dtype"]], device="cuda")
    t = whole[case["shift"]:]
    if gen is not None:
        _fill(t, gen)
    return t


def _block_sizes(case):
    """Lognormal(ln count, 1) quantiles clamped to 4 Mi: one size per pair of ranks, the same set for every seed."""
    n, normal = case["ranks"] ** 2, statistics.NormalDist()
    z = np.array([normal.inv_cdf((i + 0.5) / n) for i in range(n)])
    return np.clip(np.rint(case["count"] * np.exp(z)), 0, 4 << 20).astype(np.uint64)


def prepare(case, seed):
    H = _package()
    comms, stream = _communicator(case)
    p, n, coll = case["ranks"], case["count"], case["coll"]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    state = {"coll": coll, "comms": comms, "stream": stream.cuda_stream, "n": n, "op": _OP[case["op"]],
             "dtype": {"fp32": H.HCCL_DATA_TYPE_FP32, "fp16": H.HCCL_DATA_TYPE_FP16, "bf16": H.HCCL_DATA_TYPE_BFP16, "int8": H.HCCL_DATA_TYPE_INT8,
                       "int32": H.HCCL_DATA_TYPE_INT32, "int64": H.HCCL_DATA_TYPE_INT64}[case["dtype"]]}
    if coll == "all_reduce":
        sends = [_buffer(case, n, gen) for _ in range(p)]
        recvs = sends if case["in_place"] else [_buffer(case, n) for _ in range(p)]
    elif coll == "reduce_scatter":
        sends = [_buffer(case, n * p, gen) for _ in range(p)]
        recvs = [_buffer(case, n) for _ in range(p)]
    elif coll == "all_gather":
        recvs = [_buffer(case, n * p) for _ in range(p)]
        if case["in_place"]:
            sends = [recvs[r][r * n:(r + 1) * n] for r in range(p)]
            for t in sends:
                _fill(t, gen)
        else:
            sends = [_buffer(case, n, gen) for _ in range(p)]
    else:
        # which pair exchanges how much differs from seed to seed; blocks lie one behind the other on both sides
        cnt = np.random.default_rng(seed).permutation(_block_sizes(case)).reshape(p, p)
        back = np.ascontiguousarray(cnt.T)
        before = lambda c: np.cumsum(c, axis=1, dtype=np.uint64) - c  # noqa: E731
        state["tables"] = (cnt, before(cnt), back, before(back))
        sends = [_buffer(case, max(1, int(k)), gen) for k in cnt.sum(axis=1)]
        # a receiver has room for the most that any routing can send it
        room = max(1, int(np.sort(_block_sizes(case))[-p:].sum()))
        recvs = [_buffer(case, room) for _ in range(p)]
    state["sends"], state["recvs"] = sends, recvs
    state["sp"], state["rp"] = [t.data_ptr() for t in sends], [t.data_ptr() for t in recvs]
    return state


def run(state):
    H = _package()
    coll, comms, sp, rp, dt, stream = (state[k] for k in ("coll", "comms", "sp", "rp", "dtype", "stream"))
    if coll == "all_reduce":
        H.all_reduce(comms, sp, rp, state["n"], dt, state["op"], stream)
    elif coll == "reduce_scatter":
        H.reduce_scatter(comms, sp, rp, state["n"], dt, state["op"], stream)
    elif coll == "all_gather":
        H.all_gather(comms, sp, rp, state["n"], dt, stream)
    else:
        # a router hands over count arrays, new ones every time
        cnt, sdis, back, rdis = state["tables"]
        H.all_to_all_v(comms, sp, cnt, sdis, rp, back, rdis, dt, stream)
    return state["recvs"]


def work(case):
    p, block, unit = case["ranks"], case["count"] * _UNIT[case["dtype"]], _UNIT[case["dtype"]]
    coll = case["coll"]
    if coll == "all_reduce":
        return {"bytes": 2 * p * block, "flops": (p - 1) * case["count"]}
    if coll == "reduce_scatter":
        return {"bytes": (p * p + p) * block, "flops": (p - 1) * p * case["count"]}
    if coll == "all_gather":
        return {"bytes": (p + p * (p - 1 if case["in_place"] else p)) * block, "flops": 0}
    return {"bytes": 2 * int(_block_sizes(case).sum()) * unit, "flops": 0}


def tolerance(case):
    return "exact"
