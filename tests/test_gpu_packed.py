"""Small collectives with packed arguments (a wave per KiB of an item), against the oracle bit for bit: every shape that has a kernel of
its own (2, 4, 8, 16 sources; chains of either operand order, trees), other numbers of sources, the edges of a wave's KiB and of a
vector, in place, off a boundary, up to and beyond the sizes where the tile kernels take over."""
import numpy as np
import pytest
import torch

import closed_forms as cf
import gpu_harness as gh
from closed_forms import BF16, FP16, FP32, INT8, INT64, MAX, MIN, PROD, SUM

pytestmark = pytest.mark.gpu
RING, MESH, RHD = 0, 4, 2      # (4: the mesh without the piece cut, which these types and operations run)
MIB = 1 << 20
LIMIT = {2: 48 * MIB, 3: 7 * MIB // 2, 4: 6 * MIB, 7: 9 * MIB // 4, 8: 11 * MIB // 4, 16: 11 * MIB // 4}     # of an all-reduce; more ranks: 1.5 MiB


def _ins(dt, p, n, seed, special):
    rng = np.random.default_rng(seed)
    ins = [cf.random_input(dt, n, rng) for _ in range(p)]
    if special:
        odd = np.array([np.nan, 0.0, -0.0, np.inf, -np.inf, 1.0], np.float32)
        for x in ins:
            at = rng.random(n) < 0.5
            x[at] = cf.narrow(dt, odd[rng.integers(0, odd.size, int(at.sum()))])
    return ins


@pytest.mark.parametrize("p,algo", [(2, RING), (3, RING), (4, RING), (4, MESH), (4, RHD), (7, MESH), (8, RING), (8, MESH), (8, RHD), (11, RING), (16, RING),
                                    (16, MESH), (16, RHD), (24, RING), (32, MESH), (32, RHD)])
def test_all_reduce(orc, p, algo):
    g = gh.Group(p, algo={RING: "ring", MESH: "mesh", RHD: "rhd"}[algo])
    try:
        for k, (dt, op, pad, in_place, special) in enumerate([(FP32, SUM, 0, False, False), (BF16, MAX, 2, True, True), (FP16, MIN, 6, False, True), (INT8, SUM, 1, True, False)]):
            unit = gh.H.DTYPE_SIZE[dt]
            sizes = {1, 1024 * p // unit, 1024 * p // unit + 1, (2048 * p - 128) // unit - 1, 8 * 1024 * p // unit + 3}
            if k % 2 == (algo == RING):
                limit = min(LIMIT.get(p, 3 * MIB // 2), 4 * MIB)
                sizes |= {limit // unit - 1, limit // unit, limit // unit + 1}
            for n in sorted(sizes):
                print("packed all-reduce", p, algo, "type", dt, "op", op, "n", n, flush=True)
                ins = _ins(dt, p, n, 13 * p + n % 1013 + k, special)
                want = orc.allreduce(ins, dt, op, algo=algo)
                outs, keep = gh.all_reduce(g, ins, dt, op, in_place=in_place, pad=pad)
                assert g.info()["launches"] == 1 and g.info()["fused"] == 1
                assert g.info()["direct"] == int(n * unit <= MIB)
                for r in range(p):
                    assert gh.same(dt, outs[r], want[r]), (dt, op, n, r)
                    assert keep is None or np.array_equal(keep[r].view(np.uint8), ins[r].view(np.uint8))
    finally:
        g.close()


@pytest.mark.parametrize("p,algo", [(p, a) for p in (2, 4, 8, 16) for a in ("ring", "mesh", "rhd")])
def test_four_vectors_per_lane(orc, p, algo):
    """Between 2 and 8 MiB (16 ranks: from 1.5 MiB): whole waves of 4 KiB, one vector and one element more or less, either end of the range."""
    g = gh.Group(p, algo=algo)
    first = (3 if p == 16 else 4) * MIB // 2
    try:
        for k, (dt, op, pad, in_place, special) in enumerate([(FP32, MAX, 4, True, True), (BF16, SUM, 0, False, False), (INT8, PROD, 1, False, False), (INT64, SUM, 0, True, False)]):
            unit = gh.H.DTYPE_SIZE[dt]
            whole = (first // p + 4096) // 4096 * 4096 * p
            sizes = {whole, whole + 16 * p, whole - 16 * p} if k % 2 else {first + unit, whole + unit, whole - unit}
            if k == ("ring", "mesh", "rhd").index(algo):
                sizes |= {11 * MIB // 2 // unit * unit} if p > 4 else {6 * MIB}
            for size in sorted(sizes):
                n = size // unit
                print("packed, four vectors per lane", p, algo, "type", dt, "op", op, "n", n, flush=True)
                ins = _ins(dt, p, n, 17 * p + n % 1013 + k, special)
                want = orc.allreduce(ins, dt, op, algo={"ring": RING, "mesh": MESH, "rhd": RHD}[algo])
                outs, keep = gh.all_reduce(g, ins, dt, op, in_place=in_place, pad=pad)
                assert g.info()["launches"] == 1 and g.info()["fused"] == 1
                for r in range(p):
                    assert gh.same(dt, outs[r], want[r]), (dt, op, n, r)
                    assert keep is None or np.array_equal(keep[r].view(np.uint8), ins[r].view(np.uint8))
    finally:
        g.close()


@pytest.mark.parametrize("p", [2, 4, 5, 8, 16])
def test_blocks(orc, p):
    g = gh.Group(p)
    limit = {2: 15 * MIB, 4: 15 * MIB // 2, 8: 6 * MIB, 16: 11 * MIB // 4}.get(p, 9 * MIB // 2)
    try:
        for dt, op, pad in ((INT8, PROD, 1), (BF16, SUM, 2), (FP32, MIN, 0), (INT64, SUM, 8)):
            unit = gh.H.DTYPE_SIZE[dt]
            even = limit // p // unit // 16 * 16
            for n in (1, 1024 // unit, 1024 // unit + 1, 3 * 1024 // unit - 1) + ((even, even + 16) if dt in (BF16, FP32) else (7 * MIB // 2 // p // unit // 16 * 16 - 1,)):
                print("packed blocks", p, "type", dt, "n", n, flush=True)
                ins = _ins(dt, p, n * p, 71 * p + n, False)
                want = orc.reducescatter(ins, dt, op)
                outs, _ = gh.reduce_scatter(g, ins, dt, op, pad=pad)
                for r in range(p):
                    assert gh.same(dt, outs[r], want[r]), ("reduce-scatter", dt, n, r)
                if n < 5000:
                    parts = [x[:n] for x in ins]
                    outs = gh.all_gather(g, parts, dt, pad=pad)
                    for r in range(p):
                        assert np.array_equal(outs[r].view(np.uint8), np.concatenate(parts).view(np.uint8)), ("all-gather", dt, n, r)
    finally:
        g.close()


@pytest.mark.parametrize("p", [9, 15, 16, 17, 24, 25, 31, 32])
def test_many_sources(orc, p):
    """More than 8 sources: KiB that go to the XCDs in fours (whole groups of 32, and what is left of one), two batches of sources in flight."""
    groups = {a: gh.Group(p, algo=a) for a in ("ring", "mesh")}
    if p in (16, 24):
        groups["rhd"] = gh.Group(p, algo="rhd")
    try:
        for k, (dt, op, pad, special) in enumerate([(FP32, SUM, 0, False), (BF16, MIN, 2, True), (FP16, MAX, 6, True), (INT8, SUM, 1, False)]):
            unit = gh.H.DTYPE_SIZE[dt]
            for size in (32 * 1024 - 16, 32 * 1024, 32 * 1024 + 16 * (k % 2) + unit, 65 * 1024 + 48 + unit):
                n = size // unit
                for name, g in groups.items():
                    algo = {"ring": RING, "mesh": MESH, "rhd": RHD}[name]
                    print("many sources", p, name, "type", dt, "n", n, flush=True)
                    ins = _ins(dt, p, n * p, 5 * p + n % 811 + k, special)
                    want = orc.reducescatter(ins, dt, op, algo=algo)
                    outs, _ = gh.reduce_scatter(g, ins, dt, op, pad=pad)
                    assert g.info()["direct"] == 1 and g.info()["launches"] == 1
                    for r in range(p):
                        assert gh.same(dt, outs[r], want[r]), ("reduce-scatter", name, dt, n, r)
                    parts = [x[:n] for x in ins]
                    root = n % p
                    src, dst = [gh.to_dev(x, pad) for x in parts], [gh.empty_dev(n * unit, pad) for _ in range(p)]
                    torch.cuda.synchronize()
                    gh.H.reduce(g.comms, [t.data_ptr() for t in src], [t.data_ptr() for t in dst], n, dt, op, root, g.stream_ptr)
                    g.stream.synchronize()
                    assert g.info()["direct"] == 1 and g.info()["launches"] == 1
                    assert gh.same(dt, gh.to_host(dst[root], dt), orc.reduce_to_root(parts, dt, op, root, algo=algo)), ("reduce", name, dt, n)
                    if size < 33 * 1024 and name == "ring":
                        whole = [x[:min(n * p, MIB // unit)] for x in ins]     # (an item of every rank's, as in the others)
                        want = orc.allreduce(whole, dt, op, algo=algo)
                        outs, _ = gh.all_reduce(g, whole, dt, op, pad=pad)
                        for r in range(p):
                            assert gh.same(dt, outs[r], want[r]), ("all-reduce", dt, n, r)
    finally:
        for g in groups.values():
            g.close()


# What a call's kernels work from (HcclAmdOpForm), by quarters of a MiB on 256 CUs: up to (the first), then beyond it.
TABLES, RECORDS, PACKED, WIDE = 0, 1, 2, 3
ALL_REDUCE = {2: [(8, PACKED), (32, WIDE), (192, PACKED)], 4: [(8, PACKED), (24, WIDE), (32, TABLES), (96, PACKED)],
              8: [(8, PACKED), (11, WIDE), (16, TABLES), (22, WIDE), (32, TABLES), (48, PACKED)], 16: [(6, PACKED), (11, WIDE), (16, TABLES), (22, WIDE)]}
ALL_REDUCE_HALVES = {**ALL_REDUCE, 16: [(6, PACKED), (16, TABLES), (22, WIDE)]}
WHOLE_BLOCKS = {2: [(60, PACKED), (64, TABLES), (256, PACKED)], 3: [(24, PACKED)], 4: [(30, PACKED), (32, TABLES), (44, PACKED)], 6: [(18, PACKED)],
                8: [(24, PACKED)], 16: [(11, PACKED), (17, TABLES), (20, PACKED)]}
RAGGED_BLOCKS = {2: [(56, PACKED)], 3: [(24, PACKED)], 4: [(24, PACKED)], 6: [(16, PACKED)], 8: [(20, PACKED)], 16: [(16, PACKED)]}


def _as_the_tiles(g, call, form, what):
    """`call` takes this form and gives the bits of the tile kernels."""
    print("form", *what, "expected", form, flush=True)
    outs = call()
    assert gh.H.last_op_form(g.comms[0]) == form, what
    g.set(direct=0)
    tiles = call()
    assert gh.H.last_op_form(g.comms[0]) == TABLES
    g.set(direct="auto")
    for a, b in zip(outs, tiles):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8)), what


def _lines(edges):
    return [(upto, form, beyond) for (upto, form), (_, beyond) in zip(edges, edges[1:] + [(None, TABLES)])]


@pytest.mark.parametrize("p,algo", [(p, a) for p in (2, 4, 8, 16) for a in ("ring", "mesh", "rhd")])
def test_form_of_all_reduce(p, algo):
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256
    g = gh.Group(p, algo=algo)
    try:
        for dt, op in ((FP32, SUM), (BF16, MAX), (INT8, MIN)):
            unit = gh.H.DTYPE_SIZE[dt]
            for upto, form, beyond in _lines((ALL_REDUCE_HALVES if dt == BF16 else ALL_REDUCE)[p]):
                if upto > 100 and dt != FP32:
                    continue
                for n, want in ((upto * MIB // 4 // unit, form), (upto * MIB // 4 // unit + 1, beyond)):
                    ins = _ins(dt, p, n, 19 * p + unit, False)
                    _as_the_tiles(g, lambda: gh.all_reduce(g, ins, dt, op)[0], want, (p, algo, dt, n))
    finally:
        g.close()


@pytest.mark.parametrize("p", [2, 3, 4, 6, 8, 16])
def test_form_of_reduce_scatter(p):
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256
    g = gh.Group(p)
    try:
        for edges, ragged in ((WHOLE_BLOCKS[p], 0), (RAGGED_BLOCKS[p], 1)):
            for upto, form, beyond in _lines(edges):
                last = upto * MIB // 4 // p // 16 * 4 - 3 * ragged
                for n, want in ((last, form), (last + 4 + 12 * ragged, beyond)):
                    ins = _ins(FP32, p, n * p, 23 * p + ragged, False)
                    _as_the_tiles(g, lambda: gh.reduce_scatter(g, ins, FP32, SUM)[0], want, (p, n))
    finally:
        g.close()


def test_form_of_others():
    g = gh.Group(8, servers=2)
    try:
        ins = _ins(FP32, 8, 5000, 3, False)
        _as_the_tiles(g, lambda: gh.all_reduce(g, ins, FP32, SUM)[0], RECORDS, ("two servers",))
        g.set(servers=1)
        _as_the_tiles(g, lambda: gh.all_gather(g, ins, FP32), PACKED, ("all-gather",))
        _as_the_tiles(g, lambda: gh.all_reduce(g, ins, FP32, SUM)[0], PACKED, ("one server",))
    finally:
        g.close()


@pytest.mark.parametrize("p,quarters,up", [(2, 12, 40), (4, 7, 20), (8, 6, 20), (16, 5, 18), (6, 6, 8), (4, 7, 80)])
def test_form_off_a_boundary(p, quarters, up):
    """All-reduces whose buffers lie off 4 bytes are packed up to a size only; those off 4 or 16 bytes stop at four tiles per CU."""
    g = gh.Group(p)
    try:
        for dt, op, pad in ((BF16, MAX, 2), (INT8, SUM, 3), (FP32, SUM, 4)):
            unit = gh.H.DTYPE_SIZE[dt]
            for q in (quarters, up):
                n = q * MIB // 4 // unit
                want = TABLES if q == up and (pad != 4 or q > 64) else None
                ins = _ins(dt, p, n, 29 * p + pad, False)
                print("off a boundary", p, "type", dt, "n", n, "pad", pad, flush=True)
                outs, _ = gh.all_reduce(g, ins, dt, op, pad=pad)
                form = gh.H.last_op_form(g.comms[0])
                assert form == TABLES if want == TABLES else form in (PACKED, WIDE), (dt, n, pad, form)
                g.set(direct=0)
                tiles, _ = gh.all_reduce(g, ins, dt, op, pad=pad)
                g.set(direct="auto")
                for r in range(p):
                    assert np.array_equal(outs[r].view(np.uint8), tiles[r].view(np.uint8)), (dt, n, r)
    finally:
        g.close()
