"""Small collectives, whose descriptors ride in the kernel arguments (one launch, 4 KiB of an item per workgroup), against the
CPU checker bit for bit: the edges of a workgroup's 4 KiB and of a 16-byte vector, every batch size of sources, trees and
stack programs, buffers at any element boundary, in place, operand order on NaNs and signed zeros, new buffers on every call
and replays of a caller's graph.  Whether a call went that way is asserted for every one of them.  Whether a call went that way is asserted for every one of them."""
import numpy as np
import pytest
import torch

import closed_forms as cf
import gpu_harness as gh
from closed_forms import BF16, FP16, FP32, INT8, INT32, INT64, MAX, MIN, PROD, SUM

pytestmark = pytest.mark.gpu
H = gh.H
RING, MESH, RHD = 0, 1, 2


def _ins(dt, p, n, seed, special=False):
    rng = np.random.default_rng(seed)
    ins = [cf.random_input(dt, n, rng) for _ in range(p)]
    if special:
        odd = np.array([np.nan, 0.0, -0.0, np.inf, -np.inf, 1.0], np.float32)
        for x in ins:
            at = rng.random(n) < 0.7
            x[at] = cf.narrow(dt, odd[rng.integers(0, odd.size, int(at.sum()))])
    return ins


def _fits(plan):
    """Whether one launch's arguments hold the plan: items, sources and destinations per item, base pointers."""
    def one(cap, items, bases):
        seen = set()
        for it in plan["fused"]:
            src = [(k, r) for k, r in enumerate(it["src"]) if r]
            tree, stack = it["kind"] == 2, it["kind"] == 3
            if (it["nleaf"] if tree else len(src)) > cap or len(it["dst"]) > cap or (stack and cap > 8) or \
                    (tree and it["nleaf"] > 2 * cap // (2 if cap <= 8 else 4) and any(k & 1 for k, _ in src)):
                return False
            if len({str(r[2:]) for _, r in src}) > 1 or len({str(r[2:]) for r in it["dst"]}) > 1:
                return False
            seen |= {tuple(r[:2]) for _, r in src} | {tuple(r[:2]) for r in it["dst"]}
        return len(plan["fused"]) <= items and len(seen) <= bases
    return plan["fusedOk"] and bool(plan["fused"]) and (one(8, 16, 16) or one(32, 32, 64))


def _fits(plan):
    """Whether one launch's arguments hold the plan: items, sources and destinations per item, base pointers."""
    def one(cap, items, bases):
        seen = set()
        for it in plan["fused"]:
            src = [(k, r) for k, r in enumerate(it["src"]) if r]
            tree, stack = it["kind"] == 2, it["kind"] == 3
            if (it["nleaf"] if tree else len(src)) > cap or len(it["dst"]) > cap or (stack and cap > 8) or \
                    (tree and it["nleaf"] > min(cap, 16) and any(k & 1 for k, _ in src)):
                return False
            if len({r[2] for _, r in src}) > 1 or len({r[2] for r in it["dst"]}) > 1:
                return False
            seen |= {tuple(r[:2]) for _, r in src} | {tuple(r[:2]) for r in it["dst"]}
        return len(plan["fused"]) <= items and len(seen) <= bases
    return plan["fusedOk"] and bool(plan["fused"]) and (one(8, 16, 16) or one(32, 32, 64))


# ring: chains of 1 ... 32 sources (batches of 16, 8 and a rest); halving-doubling: trees of 2 ... 32 leaves with and
# without second sources; several groups: stack programs, with and without the piece cut (whose items do not always fit)
@pytest.mark.parametrize("p,algo,servers,cut", [(2, RING, 1, 1), (3, RING, 1, 1), (7, RING, 1, 1), (8, RING, 1, 1), (9, RING, 1, 1), (15, RING, 1, 1),
                                                (24, RING, 1, 1), (31, RING, 1, 1), (32, RING, 1, 1), (8, MESH, 1, 1), (2, RHD, 1, 1), (6, RHD, 1, 1),
                                                (8, RHD, 1, 1), (13, RHD, 1, 1), (24, RHD, 1, 1), (32, RHD, 1, 1), (8, RHD, 2, 1), (8, RHD, 4, 1),
                                                (6, RING, 3, 1), (8, RHD, 2, 0), (8, RING, 2, 0)])
def test_all_reduce(orc, p, algo, servers, cut):
    g = gh.Group(p, algo=("ring", "mesh", "rhd")[algo], servers=servers, deterministic=cut)
    ways = []
    try:
        for k, (dt, op, pad, in_place, special) in enumerate([(FP32, SUM, 0, False, False), (BF16, MAX, 2, True, True), (INT8, PROD, 3, False, False),
                                                              (FP16, MIN, 16, False, True), (INT64, SUM, 8, True, False)]):
            unit = H.DTYPE_SIZE[dt]
            sizes = {1, 128 * p // unit + 1, (4096 * p) // unit, (4096 * p + 128) // unit - 1, (3 * 4096 + 128) * p // unit + 5, (1 << 20) // unit, (1 << 20) // unit + 1}
            uncut = int(not cut and dt != INT64 and op != PROD)
            for n in sorted(sizes):
                print("small all-reduce", p, algo, servers, "type", dt, "op", op, "n", n, "pad", pad, flush=True)
                ins = _ins(dt, p, n, 31 * p + n % 1009 + k, special)
                if servers > 1:
                    want = orc.allreduce_two_level(ins, dt, op, servers, level1=algo, atomic=bool(uncut))
                else:
                    want = orc.allreduce(ins, dt, op, algo=algo)
                outs, keep = gh.all_reduce(g, ins, dt, op, in_place=in_place, pad=pad)
                word = algo | ((servers << 8 | uncut << 16) if servers > 1 else 0)
                plan = H.describe_plan(H.COLL_ALLREDUCE, word, p, n, dt, in_place_mask=(1 << p) - 1 if in_place else 0)
                ways.append(int(n * unit <= 1 << 20 and _fits(plan)))
                assert g.info()["direct"] == ways[-1] and (ways[-1] == 0 or g.info()["launches"] == 1), (dt, op, n)
                for r in range(p):
                    assert gh.same(dt, outs[r], want[r]), (dt, op, n, r)
                    assert keep is None or np.array_equal(keep[r].view(np.uint8), ins[r].view(np.uint8))
        assert 0 in ways and 1 in ways
    finally:
        g.close()


@pytest.mark.parametrize("p", [2, 5, 8, 16, 32])
def test_blocks(orc, p):
    # reduce-scatter, all-gather, broadcast, reduce and send / receive: blocks that start at any byte
    g = gh.Group(p)
    try:
        for dt, op, pad in ((INT8, SUM, 0), (BF16, SUM, 2), (FP32, MAX, 4)):
            unit = H.DTYPE_SIZE[dt]
            for n in (1, 15, 17, 4096 // unit - 1, 4096 // unit + 1, 20011 // unit):
                print("small blocks", p, "type", dt, "n", n, flush=True)
                ins = _ins(dt, p, n * p, 77 * p + n)
                want = orc.reducescatter(ins, dt, op)
                outs, _ = gh.reduce_scatter(g, ins, dt, op, pad=pad)
                assert g.info()["direct"] == 1
                for r in range(p):
                    assert gh.same(dt, outs[r], want[r]), ("reduce-scatter", dt, n, r)
                parts = [x[:n] for x in ins]
                outs = gh.all_gather(g, parts, dt, pad=pad)
                assert g.info()["direct"] == int(p * (p + 1) * n * unit <= 20 << 20)
                for r in range(p):
                    assert np.array_equal(outs[r].view(np.uint8), np.concatenate(parts).view(np.uint8)), ("all-gather", dt, n, r)
                root = n % p
                bufs = [gh.to_dev(x, pad) for x in parts]
                dst = [gh.empty_dev(n * unit, pad) for _ in range(p)]
                torch.cuda.synchronize()
                H.reduce(g.comms, [t.data_ptr() for t in bufs], [t.data_ptr() for t in dst], n, dt, op, root, g.stream_ptr)
                assert g.info()["direct"] == 1
                H.send(g.comms[0], bufs[0].data_ptr(), n, dt, p - 1, g.stream_ptr)
                spare = gh.empty_dev(n * unit, pad)
                H.recv(g.comms[p - 1], spare.data_ptr(), n, dt, 0, g.stream_ptr)
                assert g.info()["direct"] == 1
                H.broadcast(g.comms, [t.data_ptr() for t in bufs], n, dt, root, g.stream_ptr)
                assert g.info()["direct"] == 1
                g.stream.synchronize()
                assert gh.same(dt, gh.to_host(dst[root], dt), orc.reduce_to_root(parts, dt, op, root)), ("reduce", dt, n)
                assert np.array_equal(gh.to_host(spare, dt).view(np.uint8), parts[0].view(np.uint8)), ("send / receive", dt, n)
                for r in range(p):
                    assert np.array_equal(gh.to_host(bufs[r], dt).view(np.uint8), parts[root].view(np.uint8)), ("broadcast", dt, n, r)
    finally:
        g.close()


def test_new_buffers_and_graph_replay(orc):
    p, n = 8, 3001
    g = gh.Group(p)
    try:
        ins = _ins(FP32, p, n, 5)
        want = orc.allreduce(ins, FP32, SUM)
        base = [gh.to_dev(x) for x in ins]
        sets = [([t.clone() for t in base], [torch.zeros_like(t) for t in base]) for _ in range(20)]
        torch.cuda.synchronize()
        hits = []
        for s, r in sets + sets[-1:]:
            H.all_reduce(g.comms, [t.data_ptr() for t in s], [t.data_ptr() for t in r], n, FP32, SUM, g.stream_ptr)
            hits.append(g.info()["cacheHit"])
            assert g.info()["direct"] == 1
        assert hits == [0] * 20 + [1]
        s, r = sets[3]
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(g.stream):
            graph.capture_begin()
            H.all_reduce(g.comms, [t.data_ptr() for t in s], [t.data_ptr() for t in r], n, FP32, SUM, g.stream_ptr)
            graph.capture_end()
        for replay in range(3):
            for t in r:
                t.zero_()
            H.all_reduce(g.comms, [t.data_ptr() for t in sets[7][0]], [t.data_ptr() for t in sets[7][1]], n, FP32, SUM, g.stream_ptr)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            for k in range(p):
                assert np.array_equal(gh.to_host(r[k], FP32), want[k]), (replay, k)
        for _, r in sets:
            for k in range(p):
                assert np.array_equal(gh.to_host(r[k], FP32), want[k])
    finally:
        g.close()


@pytest.mark.parametrize("p", [4, 33])
def test_overlapping_buffers_among_in_place_ranks(orc, p):
    # some ranks in place, all else apart: one pass; a send buffer that reaches into another rank's receive buffer, or into its
    # own at another offset: staged; two receive buffers that overlap: refused, and what is called next is not disturbed
    n, dt = 1000, INT8
    ins = _ins(dt, p, n, 11)
    want = orc.allreduce(ins, dt, SUM)
    g = gh.Group(p)
    try:
        for case in ("apart", "into another's", "into its own", "two receivers", "apart"):
            pool = torch.zeros(2 * p * 4096, dtype=torch.uint8, device="cuda")
            at = lambda k: pool[k * 4096:k * 4096 + n]  # noqa: E731
            sends, recvs = [at(2 * r) for r in range(p)], [at(2 * r if r % 3 == 1 else 2 * r + 1) for r in range(p)]
            if case == "into another's":
                recvs[0] = pool[4 * 4096 + n - 1:4 * 4096 + n - 1 + n]      # the last byte of rank 2's send buffer
            elif case == "into its own":
                recvs[0] = pool[1:1 + n]
            elif case == "two receivers":
                recvs[0] = pool[5 * 4096 + n - 1:5 * 4096 + n - 1 + n]              # the last byte of rank 2's receive buffer
            for r in range(p):
                sends[r].copy_(torch.from_numpy(ins[r].view(np.uint8)))
            torch.cuda.synchronize()
            args = (g.comms, [t.data_ptr() for t in sends], [t.data_ptr() for t in recvs], n, dt, SUM, g.stream_ptr)
            print("overlap", p, case, flush=True)
            if case == "two receivers":
                with pytest.raises(H.HcclError) as e:
                    H.all_reduce(*args)
                assert e.value.code == H.HCCL_E_PARA
                continue
            H.all_reduce(*args)
            g.stream.synchronize()
            assert g.info()["fused"] == (1 if case == "apart" else 0)
            for r in range(p):
                assert gh.same(dt, gh.to_host(recvs[r], dt), want[r]), (case, r)
    finally:
        g.close()


@pytest.mark.parametrize("p", [2, 8, 32])
def test_size_limits(p):
    # the largest of every collective that goes out this way, and one element more; integers, whose sums have no order
    mib = 1 << 20
    g = gh.Group(p)
    try:
        for dt in (INT8, INT32, INT64):
            unit = H.DTYPE_SIZE[dt]
            kind = {INT8: torch.int8, INT32: torch.int32, INT64: torch.int64}[dt]
            even = 16 // unit
            to_one = 4 * mib if p <= 3 or dt == INT8 else 5 * mib // 2
            cases = [("reduce_scatter", to_one // p // unit // even * even, 1), ("reduce_scatter", to_one // p // unit // even * even + even, 0),
                     ("reduce_scatter", 4 * mib // p // unit // even * even - 1, 1), ("reduce_scatter", 4 * mib // p // unit // even * even + 1, 0),
                     ("reduce", to_one // unit, 1), ("reduce", to_one // unit + even, 0), ("reduce", 4 * mib // unit - 1, 1), ("reduce", 4 * mib // unit + 1, 0),
                     ("all_gather", 20 * mib // p // (p + 1) // unit, 1), ("all_gather", 20 * mib // p // (p + 1) // unit + 1, 0),
                     ("broadcast", 20 * mib // p // unit, 1), ("broadcast", 20 * mib // p // unit + 1, 0),
                     ("scatter", 10 * mib // p // unit, 1), ("scatter", 10 * mib // p // unit + 1, 0),
                     ("send", 10 * mib // unit, 1), ("send", 10 * mib // unit + 1, 0)]
            for coll, n, direct in cases:
                if p == 32 and coll == "reduce" and dt != INT32:
                    continue
                print("limit", p, coll, "type", dt, "n", n, flush=True)
                gen = torch.Generator(device="cuda")
                gen.manual_seed(n)
                rand = lambda k: torch.randint(-100, 100, (k,), dtype=kind, device="cuda", generator=gen)  # noqa: E731
                zero = lambda k: torch.zeros(k, dtype=kind, device="cuda")  # noqa: E731
                ptr = lambda ts: [0 if t is None else t.data_ptr() for t in ts]  # noqa: E731
                root = p - 1
                if coll == "reduce_scatter":
                    s, r = [rand(n * p) for _ in range(p)], [zero(n) for _ in range(p)]
                    torch.cuda.synchronize()
                    H.reduce_scatter(g.comms, ptr(s), ptr(r), n, dt, SUM, g.stream_ptr)
                    want = list(sum(s[1:], s[0].clone()).split(n))
                elif coll == "reduce":
                    s, r = [rand(n) for _ in range(p)], [zero(n) for _ in range(p)]
                    torch.cuda.synchronize()
                    H.reduce(g.comms, ptr(s), ptr(r), n, dt, SUM, root, g.stream_ptr)
                    r, want = [r[root]], [sum(s[1:], s[0].clone())]
                elif coll == "all_gather":
                    s, r = [rand(n) for _ in range(p)], [zero(n * p) for _ in range(p)]
                    torch.cuda.synchronize()
                    H.all_gather(g.comms, ptr(s), ptr(r), n, dt, g.stream_ptr)
                    want = [torch.cat(s)] * p
                elif coll == "broadcast":
                    r = [rand(n) for _ in range(p)]
                    want = [r[root].clone()] * p
                    torch.cuda.synchronize()
                    H.broadcast(g.comms, ptr(r), n, dt, root, g.stream_ptr)
                elif coll == "scatter":
                    s, r = [None] * root + [rand(n * p)], [zero(n) for _ in range(p)]
                    torch.cuda.synchronize()
                    H.scatter(g.comms, ptr(s), ptr(r), n, dt, root, g.stream_ptr)
                    want = list(s[root].split(n))
                else:
                    s, r = [rand(n)], [zero(n)]
                    torch.cuda.synchronize()
                    H.send(g.comms[0], s[0].data_ptr(), n, dt, root, g.stream_ptr)
                    H.recv(g.comms[root], r[0].data_ptr(), n, dt, 0, g.stream_ptr)
                    want = s
                g.stream.synchronize()
                assert g.info()["direct"] == direct, (coll, n)
                for a, b in zip(r, want):
                    assert torch.equal(a, b), (coll, n)
    finally:
        g.close()
