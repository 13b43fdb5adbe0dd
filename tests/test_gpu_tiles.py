"""Whole tiles and what is left behind them: rounds of one to eight tiles of a team, borders between items inside a round,
pieces shorter than a tile, element-wise ends of every number of sources, blocks of which only the sources or only the
destinations lie on a 16-byte boundary.  Against the CPU checker, bit for bit; bytes around the results untouched."""
import numpy as np
import pytest
import torch

import closed_forms as cf
import gpu_harness as gh
from closed_forms import BF16, FP16, FP32, FP64, INT8, INT64, MAX, MIN, PROD, SUM, UINT8

pytestmark = pytest.mark.gpu
H = gh.H
TILE = 16384


@pytest.fixture(scope="module")
def orc():
    from oracle import oracle
    oracle.build()
    return oracle


def _ins(dt, p, n, seed):
    rng = np.random.default_rng(seed)
    return [cf.random_input(dt, n, rng) for _ in range(p)]


@pytest.mark.parametrize("dt,op,algo,servers", [(FP32, SUM, "ring", 1), (FP16, MAX, "ring", 1), (INT8, PROD, "ring", 1), (BF16, SUM, "rhd", 1), (FP32, MIN, "auto", 2)])
def test_rounds_of_one_to_eight_tiles(orc, dt, op, algo, servers):
    # 8 ranks: n tiles for each of 256 workgroups make one round; slices of odd lengths put item borders inside it
    p = 8
    g = gh.Group(p, algo=algo, servers=servers, team=1)
    try:
        for tiles in (1, 2, 3, 4, 5, 6, 7, 8, 9):
            n = (256 * tiles * TILE - 37 * TILE) // H.DTYPE_SIZE[dt] + 5
            print("round of", tiles, "type", dt, "op", op, algo, flush=True)
            ins = _ins(dt, p, n, 9800 + tiles)
            if servers == 2:
                want = orc.allreduce_two_level(ins, dt, op, 2, level1=orc.RHD, atomic=True, threads=8)
            else:
                want = orc.allreduce([x.copy() for x in ins], dt, op, algo={"ring": 0, "rhd": 2}[algo], threads=8)
            outs, _ = gh.all_reduce(g, ins, dt, op, pad=6 if dt == FP16 else 0)
            assert g.info()["teamLaunches"] >= 1
            for r in range(p):
                assert gh.same(dt, outs[r], want[r]), (tiles, r)
    finally:
        g.close()


@pytest.mark.parametrize("p", [8, 3])
def test_gathered_rounds(p):
    # one source, many destinations: blocks that start at every byte
    g = gh.Group(p, algo="ring", team=1)
    try:
        for tiles in (1, 2, 4, 7, 8, 9):
            n = 256 * tiles * TILE // p + 1001
            print("gathered rounds", p, tiles, n, flush=True)
            ins = _ins(INT8, p, n, 9900 + tiles)
            outs = gh.all_gather(g, ins, INT8)
            assert g.info()["teamLaunches"] >= 1
            want = np.concatenate(ins)
            for r in range(p):
                assert np.array_equal(outs[r], want), (tiles, r)
    finally:
        g.close()


@pytest.mark.parametrize("dt,op", [(FP32, MIN), (BF16, MAX), (INT8, SUM), (UINT8, MAX), (INT64, PROD), (FP16, SUM)])
def test_short_blocks_of_any_number_of_sources(orc, dt, op):
    # element-wise ends, pieces of less and more than a vector per lane, both chain kernels (results with one destination and
    # with several), trees with and without second sources
    for p in (2, 3, 5, 7, 8, 9, 11, 12, 13, 16, 17, 24, 32):
        for algo in ("ring", "rhd"):
            g = gh.Group(p, algo=algo, team=0, direct=0)
            try:
                for n in (1, 7, 61, 1021, 5003, 20011):
                    print("short blocks", dt, op, p, algo, n, flush=True)
                    ins = _ins(dt, p, n * p, 9100 + n)
                    want = orc.reducescatter(ins, dt, op, algo={"ring": 0, "rhd": 2}[algo])
                    outs, _ = gh.reduce_scatter(g, ins, dt, op)
                    for r in range(p):
                        assert gh.same(dt, outs[r], want[r]), (p, algo, n, r)
                    ins = _ins(dt, p, n, 9200 + n)
                    want = orc.allreduce([x.copy() for x in ins], dt, op, algo={"ring": 0, "rhd": 2}[algo])
                    outs, _ = gh.all_reduce(g, ins, dt, op)
                    for r in range(p):
                        assert gh.same(dt, outs[r], want[r]), (p, algo, n, r)
            finally:
                g.close()


@pytest.mark.parametrize("team", [0, 1])
@pytest.mark.parametrize("dt,op,offsets", [(FP16, MAX, (0, 2, 2, 2, 6, 0)), (INT8, SUM, (1, 1, 1, 3, 0, 5)), (FP32, SUM, (4, 0, 0, 0, 8, 12)), (BF16, SUM, (2, 4, 6, 8, 10, 12))])
def test_buffers_at_different_offsets(orc, dt, op, offsets, team):
    # the pointers of an item agree in part, or not at all
    p, unit = len(offsets), H.DTYPE_SIZE[dt]
    g = gh.Group(p, algo="ring", team=team, direct=0)
    try:
        for n in (3, 6 * TILE // unit + 11, 50 * TILE // unit + 3):
            print("offsets", dt, op, team, n, flush=True)
            ins = _ins(dt, p, n, 9300 + n)
            want = orc.allreduce([x.copy() for x in ins], dt, op)
            sends = [gh.to_dev(x, 16 + o) for x, o in zip(ins, offsets)]
            whole = [torch.full((n * unit + 64,), 0xA5, dtype=torch.uint8, device="cuda") for _ in ins]
            at = [16 + offsets[(r + 2) % p] for r in range(p)]
            torch.cuda.synchronize()
            H.all_reduce(g.comms, [t.data_ptr() for t in sends], [t.data_ptr() + at[r] for r, t in enumerate(whole)], n, dt, op, g.stream_ptr)
            g.stream.synchronize()
            for r in range(p):
                t = whole[r]
                assert gh.same(dt, gh.to_host(t[at[r]:at[r] + n * unit].clone(), dt), want[r]), (n, r)
                assert bool((t[:at[r]] == 0xA5).all()) and bool((t[at[r] + n * unit:] == 0xA5).all()), (n, r)
    finally:
        g.close()


@pytest.mark.parametrize("dt,op", [(FP32, SUM), (BF16, MAX), (INT8, SUM)])
@pytest.mark.parametrize("algo", ["ring", "mesh"])
def test_steps_with_only_the_destination_off(orc, dt, op, algo):
    # step by step, both operands at one offset from a 16-byte boundary and the destination at another
    p, unit = 4, H.DTYPE_SIZE[dt]
    g = gh.Group(p, algo=algo, fuse=0, deterministic=1)
    try:
        for n, src, dst in ((5, 0, unit), (3 * TILE // unit + 7, 0, unit), (3 * TILE // unit + 7, unit, 0), (7 * TILE // unit + 1, 8, 8 + unit)):
            print("steps", dt, op, algo, n, src, dst, flush=True)
            ins = _ins(dt, p, n * p, 9500 + n)
            want = orc.reducescatter(ins, dt, op, algo={"ring": 0, "mesh": 1}[algo])
            sends = [gh.to_dev(x, 16 + src) for x in ins]
            whole = [torch.full((n * unit + 64,), 0xA5, dtype=torch.uint8, device="cuda") for _ in ins]
            torch.cuda.synchronize()
            H.reduce_scatter(g.comms, [t.data_ptr() for t in sends], [t.data_ptr() + 16 + dst for t in whole], n, dt, op, g.stream_ptr)
            g.stream.synchronize()
            assert g.info()["fused"] == 0
            for r in range(p):
                t = whole[r]
                assert gh.same(dt, gh.to_host(t[16 + dst:16 + dst + n * unit].clone(), dt), want[r]), (n, r)
                assert bool((t[:16 + dst] == 0xA5).all()) and bool((t[16 + dst + n * unit:] == 0xA5).all()), (n, r)
    finally:
        g.close()


@pytest.mark.parametrize("dt,op", [(FP16, MAX), (FP16, MIN), (BF16, MAX), (BF16, MIN)])
@pytest.mark.parametrize("p,team", [(8, 0), (8, 1), (5, 0), (2, 1), (12, 0)])
def test_half_selection_over_every_bit_pattern(orc, dt, op, p, team):
    # NaNs of every payload, both zeros, infinities, denormals: most waves see one, some results are zeros of either sign
    g = gh.Group(p, algo="ring", team=team, direct=0)
    try:
        for n, kind in ((70001, "any"), (70001, "zeros"), (300007, "rare")):
            print("selection", dt, op, p, team, n, kind, flush=True)
            rng = np.random.default_rng(9400 + n + p)
            ins = []
            for r in range(p):
                if kind == "any":
                    x = rng.integers(0, 1 << 16, n, dtype=np.uint16)
                elif kind == "zeros":
                    x = rng.choice(np.array([0x0000, 0x8000, 0x0001, 0x8001, 0x3c00 if op == MIN else 0xbc00], np.uint16), n)
                else:
                    x = cf.random_input(dt, n, rng)
                    x[rng.integers(0, n, 5)] = rng.choice(np.array([0x7fc1, 0xffff, 0x7c01, 0x7f81, 0x0000, 0x8000, 0x7f80, 0xff80, 0x7c00, 0xfc00], np.uint16), 5)
                ins.append(x)
            want = orc.allreduce([x.copy() for x in ins], dt, op)
            for in_place in (False, True):
                outs, _ = gh.all_reduce(g, ins, dt, op, in_place=in_place)
                for r in range(p):
                    assert np.array_equal(outs[r].view(np.uint16), want[r].view(np.uint16)), (kind, in_place, r)
    finally:
        g.close()


def _placed_specials(dt, op, p, rng):
    """Ordinary values, and every 2600 elements (a wave reads 2048 of a tile) one place where up to two sources hold a special
    one, in each half of a word, in the first, a middle and the last source."""
    inf = 0x7f80 if dt == BF16 else 0x7c00
    singles = [inf, 0x8000 | inf, inf | 0x40 if dt == BF16 else inf | 0x200, 0x8000 | inf | 1, inf | 1, 0x0000, 0x8000, 0x0001, 0x8001]
    places = sorted({0, p // 2, p - 1})
    kinds = [[(v, r)] for v in singles for r in places]
    kinds += [[(a, r), (b, q)] for a, b in ((0x0000, 0x8000), (0x8000, 0x0000)) for r in places for q in places if r < q]
    step = 2600
    n = 2 * step * len(kinds)
    # losing values: a zero placed among them is the result
    lose = rng.integers(1, 0x30, n).astype(np.uint16) * 0x100 + rng.integers(0, 256, n).astype(np.uint16)
    ins = [np.roll(lose, 17 * r) | np.uint16(0x8000 if op == MAX else 0) for r in range(p)]
    for i, kind in enumerate(kinds):
        for half in (0, 1):
            at = (2 * i + half) * step + int(rng.integers(0, step // 2)) * 2 + half
            for v, r in kind:
                ins[r][at] = v
    return ins


@pytest.mark.parametrize("dt,op", [(FP16, MAX), (FP16, MIN), (BF16, MAX), (BF16, MIN)])
@pytest.mark.parametrize("team", [0, 1])
def test_half_selection_with_one_special_in_a_wave(orc, dt, op, team):
    # the result of the fast fold stands in most waves: it may be a zero of either sign, an infinity, a denormal
    for p in range(2, 10):
        g = gh.Group(p, algo="ring", team=team, direct=0)
        try:
            print("placed specials", dt, op, p, team, flush=True)
            ins = _placed_specials(dt, op, p, np.random.default_rng(9600 + p))
            want = orc.allreduce([x.copy() for x in ins], dt, op)
            outs, _ = gh.all_reduce(g, ins, dt, op)
            for r in range(p):
                assert np.array_equal(outs[r].view(np.uint16), want[r].view(np.uint16)), (p, r)
        finally:
            g.close()


@pytest.mark.parametrize("dt,op", [(FP32, MAX), (FP32, MIN), (FP64, MAX)])
@pytest.mark.parametrize("algo", ["ring", "mesh"])
def test_rounds_keep_the_operand_order(orc, dt, op, algo):
    # rounds read source by source whose tiles belong to two items, on values that tell the order: zeros of both signs, NaNs
    p, unit = 8, H.DTYPE_SIZE[dt]
    bits = np.uint32 if unit == 4 else np.uint64
    top = 32 if unit == 4 else 64
    exp = 0x7f800000 if unit == 4 else 0x7ff0000000000000
    values = np.array([0, 1 << (top - 1), 0, 1 << (top - 1), exp | 1, exp | (1 << (top - 1)) | 77, 1, exp], bits)
    g = gh.Group(p, algo=algo, team=1)
    try:
        for tiles in (4, 5, 6, 7, 8):
            n = (256 * tiles * TILE - 37 * TILE) // unit + 5
            print("order in rounds of", tiles, "type", dt, "op", op, algo, flush=True)
            rng = np.random.default_rng(9700 + tiles)
            ins = [values[rng.integers(0, len(values), n)].view(np.float32 if unit == 4 else np.float64) for _ in range(p)]
            want = orc.allreduce([x.copy() for x in ins], dt, op, algo={"ring": orc.RING, "mesh": orc.MESH_ATOMIC}[algo], threads=8)
            outs, _ = gh.all_reduce(g, ins, dt, op)
            assert g.info()["teamLaunches"] >= 1
            for r in range(p):
                assert np.array_equal(outs[r].view(bits), want[r].view(bits)), (tiles, r)
    finally:
        g.close()
