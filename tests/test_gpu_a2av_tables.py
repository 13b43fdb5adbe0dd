"""All-to-all-v straight from the callers' tables (csrc/a2av.cc, kernels_a2av.h) against its definition, byte for byte, whole receive buffers
with what lies between the blocks: rank counts around the kernels' 8, 16, 32, 64, element sizes, empty blocks, blocks at any byte, blocks in
any order with gaps, pieces at the edges of 4 KiB, several sets of tables and streams in turn, and the calls that go the general way."""
import ctypes
import threading

import numpy as np
import pytest
import torch

import gpu_harness as gh

pytestmark = pytest.mark.gpu
H = gh.H
TYPES = {1: H.HCCL_DATA_TYPE_INT8, 2: H.HCCL_DATA_TYPE_BFP16, 4: H.HCCL_DATA_TYPE_INT32, 8: H.HCCL_DATA_TYPE_INT64, 16: H.HCCL_DATA_TYPE_INT128}


def _tables(rng, p, sizes, order="packed"):
    """count, send displacement, receive count, receive displacement; elements in all of every rank's buffers."""
    cnt = sizes(p).astype(np.int64)
    sd, rd = np.zeros((p, p), np.int64), np.zeros((p, p), np.int64)
    for r in range(p):
        for table, lens in ((sd, cnt[r]), (rd, cnt[:, r])):
            at = 0
            for k in (range(p) if order == "packed" else rng.permutation(p)):
                at += 0 if order == "packed" else int(rng.integers(0, 5))
                table[r, k] = at
                at += int(lens[k])
    room = [int(max([0] + [t[r, k] + n for k, n in enumerate(lens)])) for t, c in ((sd, cnt), (rd, cnt.T)) for r, lens in enumerate(c)]
    return [np.ascontiguousarray(x).astype(np.uint64) for x in (cnt, sd, cnt.T, rd)], room[:p], room[p:]


class Run:
    """Buffers and tables of one call, and what it has to write."""

    def __init__(self, rng, p, unit, sizes, order="packed", pad=0):
        self.p, self.unit = p, unit
        self.t, sroom, rroom = _tables(rng, p, sizes, order)
        self.sends = [rng.integers(0, 256, max(1, n) * unit, dtype=np.uint8) for n in sroom]
        self.dev = [torch.from_numpy(np.concatenate([np.zeros(pad, np.uint8), x])).cuda() for x in self.sends]
        self.pad = pad
        self.out = [torch.empty(pad + n * unit + 64, dtype=torch.uint8, device="cuda") for n in rroom]

    def call(self, g, stream=None, t=None):
        H.all_to_all_v(g.comms, [x.data_ptr() + self.pad for x in self.dev], *(t or self.t)[:2], [x.data_ptr() + self.pad for x in self.out], *(t or self.t)[2:],
                       TYPES[self.unit], g.stream_ptr if stream is None else stream.cuda_stream)

    def clear(self):
        for o in self.out:
            o.fill_(0xA5)
        torch.cuda.synchronize()

    def check(self):
        torch.cuda.synchronize()
        cnt, sd, _, rd = (x.astype(np.int64) * self.unit for x in self.t)
        for j in range(self.p):
            want = np.full(self.out[j].numel(), 0xA5, np.uint8)
            for i in range(self.p):
                want[self.pad + rd[j, i]:self.pad + rd[j, i] + cnt[i, j]] = self.sends[i][sd[i, j]:sd[i, j] + cnt[i, j]]
            assert np.array_equal(self.out[j].cpu().numpy(), want), j


@pytest.mark.parametrize("p", [1, 2, 7, 8, 9, 16, 17, 32, 33, 64])
def test_shapes(p):
    rng = np.random.default_rng(4200 + p)
    g = gh.Group(p)
    try:
        short = lambda n: rng.integers(0, 40, (n, n)) * (rng.random((n, n)) < 0.7)  # noqa: E731
        skewed = lambda n: np.minimum(np.exp(rng.normal(4.5, 2.0, (n, n))), 40000)  # noqa: E731
        edges = lambda n: rng.choice([0, 1, 15, 16, 17, 127, 128, 129, 4095, 4096, 4097, 8191, 8192, 8193], (n, n))  # noqa: E731
        nothing = lambda n: np.zeros((n, n))  # noqa: E731
        one = lambda n: (np.arange(n * n).reshape(n, n) == n * n - 1) * 5000  # noqa: E731
        for unit, sizes, order, pad in ((1, edges, "packed", 0), (1, short, "any", 3), (2, skewed, "any", 6), (4, skewed, "packed", 0), (4, short, "any", 4),
                                        (8, edges, "any", 8), (16, short, "packed", 16), (4, nothing, "packed", 0), (4, one, "packed", 4)):
            print("tables", p, "unit", unit, order, "pad", pad, flush=True)
            run = Run(rng, p, unit, sizes, order, pad)
            for again in range(2):
                run.clear()
                run.call(g)
                run.check()
                info = g.info()
                assert (info["cacheHit"], info["fused"], info["scratchBytes"]) == (again, 1, 0)
                total = int(run.t[0].sum()) * unit
                assert info["launches"] == (1 if total else 0) and info["bytesRead"] == info["bytesWritten"] == info["schedRead"] == total
    finally:
        g.close()


@pytest.mark.parametrize("p,mib", [(8, 40), (16, 40), (4, 600), (32, 48), (8, 100), (16, 100), (32, 100), (48, 140)])
def test_large(p, mib):
    # beyond 96 MiB in all workgroups of four waves, beyond 256 MiB several launches
    rng = np.random.default_rng(77)
    g = gh.Group(p)
    try:
        run = Run(rng, p, 2, lambda n: rng.dirichlet(np.ones(n * n)).reshape(n, n) * (mib << 19), "packed", 2)
        for _ in range(2):      # (a new call, a known one)
            run.clear()
            run.call(g)
            run.check()
        total = int(run.t[0].sum()) * 2
        assert g.info()["launches"] == -(-total // (256 << 20))
    finally:
        g.close()


@pytest.mark.parametrize("p", [5, 20])
def test_sets_and_streams_in_turn(p):
    rng = np.random.default_rng(31 + p)
    g = gh.Group(p)
    try:
        runs = [Run(rng, p, 4, lambda n: rng.integers(0, 300, (n, n)), "any", 4) for _ in range(11)]     # more than are kept
        streams = [g.stream, torch.cuda.Stream(), torch.cuda.Stream()]
        for turn in range(3):
            for r in runs:
                r.clear()
            for k, r in enumerate(runs):
                r.call(g, streams[(k + turn) % len(streams)])
            for r in runs:
                r.check()
        # tables that part late: only the last rank's rows differ, and back again
        a = runs[0]
        b = Run(rng, p, 4, lambda n: a.t[0].astype(np.int64), "packed", 4)
        b.t = [x.copy() for x in a.t]
        b.t[3][p - 1] += np.uint64(2)
        b.sends, b.dev = a.sends, a.dev
        b.out = [torch.empty(o.numel() + 16, dtype=torch.uint8, device="cuda") for o in a.out]
        for r in (a, b, a, b, b):
            r.clear()
            r.call(g)
            r.check()
        assert g.info()["cacheHit"] == 1
    finally:
        g.close()


@pytest.mark.parametrize("p", [10, 24])
def test_no_stream_waits_for_another(p):
    """A call known by its numbers is known on every stream; new tables on streams in turn are queued while another stream is at work."""
    rng = np.random.default_rng(83 + p)
    g = gh.Group(p)
    try:
        runs = [Run(rng, p, 4, lambda n: rng.integers(0, 300, (n, n)), "any", 4) for _ in range(16)]
        streams = [torch.cuda.Stream() for _ in range(3)]
        for r in runs:
            r.clear()
        for k, r in enumerate(runs[:10]):       # (more than are kept, on all of the streams)
            r.call(g, streams[k % 3])
        torch.cuda.synchronize()
        for r in runs[:10]:
            r.check()
        for r in runs[4:10]:
            r.clear()
        for r in runs[4:10]:
            for s in streams:
                r.call(g, s)
                assert g.info()["cacheHit"] == 1
        for r in runs[4:10]:
            r.check()
        busy, there = torch.cuda.Stream(), torch.cuda.Event()
        with torch.cuda.stream(busy):
            torch.cuda._sleep(200_000_000)
            there.record()
        for k, r in enumerate(runs[10:16]):     # (no more than there are pinned buffers for them)
            r.call(g, streams[(2 * k) % 3])
            assert g.info()["cacheHit"] == 0
        assert not there.query(), "a call waited for work on another stream"
        for r in runs[10:16]:
            r.check()
    finally:
        g.close()


@pytest.mark.parametrize("p", [6, 18])
def test_the_general_way_gives_the_same(p):
    rng = np.random.default_rng(59 + p)
    g = gh.Group(p)
    try:
        run = Run(rng, p, 4, lambda n: rng.integers(0, 900, (n, n)) * (rng.random((n, n)) < 0.8), "any", 4)
        infos = []
        for params in ({"direct": "auto"}, {"direct": "0"}, {"direct": "auto", "servers": 2}, {"direct": "0", "servers": 2}, {"direct": "auto", "servers": 1, "fuse": 0}):
            g.set(**params)
            run.clear()
            run.call(g)
            run.check()
            infos.append({k: v for k, v in g.info().items() if k not in ("launches", "cacheHit", "graph")})
        assert infos[0] == infos[1] and infos[2] == infos[3]
        g.set(fuse=1)
        # a displacement beyond 32 bits where nothing is sent
        i, j = np.argwhere(run.t[0] == 0)[0]
        far = [x.copy() for x in run.t]
        far[1][i, j] = np.uint64(1 << 40)
        for t in (far, run.t, far):
            run.clear()
            run.call(g, t=t)
            run.check()
        # the two sides disagree: refused, and what comes next is not disturbed
        bad = [x.copy() for x in run.t]
        i, j = np.argwhere(run.t[0] != 0)[-1]
        bad[0][i, j] += np.uint64(1)
        with pytest.raises(H.HcclError) as e:
            run.call(g, t=bad)
        assert e.value.code == H.HCCL_E_PARA
        run.clear()
        run.call(g)
        run.check()
        # a rank's receive buffer lies over another rank's send buffer: staged
        over = Run(rng, p, 4, lambda n: np.full((n, n), 50), "packed", 0)
        spare = torch.empty(over.dev[1].numel() + over.out[0].numel(), dtype=torch.uint8, device="cuda")
        spare[:over.dev[1].numel()] = over.dev[1]
        over.dev[1], over.out[0] = spare[:over.dev[1].numel()], spare[over.dev[1].numel() - 4:][:over.out[0].numel()]
        for r in range(1, p):
            over.out[r].fill_(0xA5)
        torch.cuda.synchronize()
        over.call(g)
        torch.cuda.synchronize()
        assert g.info()["fused"] == 0
        over.out[0][p * 50 * 4:] = 0xA5
        over.check()
        # recorded into a caller's graph, replayed between calls of its own
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(g.stream):
            graph.capture_begin()
            run.call(g)
            graph.capture_end()
        for _ in range(3):
            run.clear()
            graph.replay()
            run.check()
            run.clear()
            run.call(g)
            run.check()
    finally:
        g.close()


def test_new_tables_under_load():
    # tables in device memory: written anew while earlier calls are still under way
    p = 40
    rng = np.random.default_rng(3)
    g = gh.Group(p)
    try:
        runs = [Run(rng, p, 1, lambda n: rng.integers(0, 2000, (n, n)), "packed", 0) for _ in range(20)]
        for r in runs:
            r.clear()
        for r in runs:
            r.call(g)
        for r in runs:
            r.check()
    finally:
        g.close()


@pytest.mark.parametrize("p", [2, 8, 9, 16, 17, 32, 33, 64])
def test_which_form(p):
    """A new call, a known one, the general way (HcclAmdOpForm: 4 in the arguments, 5 in device memory, 0 planned)."""
    rng = np.random.default_rng(7 * p)
    g = gh.Group(p)
    try:
        run = Run(rng, p, 4, lambda n: rng.integers(0, 300, (n, n)), "packed", 4)
        for params, want in (({}, 4 if p <= 16 else 5), ({}, 5), ({}, 5), ({"direct": 0}, 0), ({"direct": "auto"}, 5)):
            g.set(**params)
            run.clear()
            run.call(g)
            assert H.last_op_form(g.comms[0]) == want, params
            run.check()
        n = 1000
        send, recv = [torch.randint(0, 256, (p * n,), dtype=torch.uint8, device="cuda") for _ in range(p)], [torch.empty(p * n, dtype=torch.uint8, device="cuda") for _ in range(p)]
        torch.cuda.synchronize()
        for want in (4 if p <= 16 else 5, 5):
            H.all_to_all(g.comms, [t.data_ptr() for t in send], [t.data_ptr() for t in recv], n, TYPES[1], g.stream_ptr)
            assert H.last_op_form(g.comms[0]) == want
        g.stream.synchronize()
        for j in range(p):
            assert torch.equal(recv[j], torch.cat([send[i][j * n:(j + 1) * n] for i in range(p)])), j
    finally:
        g.close()


@pytest.mark.parametrize("p", [12, 20])
def test_one_thread_and_stream_per_rank(p):
    """Whichever rank comes last, on whichever stream: a known call is known."""
    rng = np.random.default_rng(11 * p)
    g = gh.Group(p, blocking_arrive=1, arrive_timeout_ms=20000)
    try:
        runs = [Run(rng, p, 4, lambda n: rng.integers(0, 300, (n, n)), "any", 4) for _ in range(4)]
        streams = [torch.cuda.Stream() for _ in range(p)]
        for r in runs:
            r.clear()
        codes, seen = [[] for _ in range(p)], []

        def work(r):
            for turn in range(4):
                for run in runs:
                    rows = [t[r].ctypes.data for t in run.t]
                    codes[r].append(H.lib().HcclAlltoAllV(run.dev[r].data_ptr() + run.pad, rows[0], rows[1], TYPES[4], run.out[r].data_ptr() + run.pad, rows[2], rows[3],
                                                          TYPES[4], g.comms[r], streams[r].cuda_stream))
                    if r == 0 and turn:
                        seen.append(H.last_op_info(g.comms[0])["cacheHit"])
            streams[r].synchronize()

        threads = [threading.Thread(target=work, args=(r,)) for r in range(p)]
        for t in threads:
            t.start()
        for t in threads:
            t.join(60)
        assert codes == [[0] * 16] * p and seen == [1] * 12
        for r in runs:
            r.check()
    finally:
        g.close()
