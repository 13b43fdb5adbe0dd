"""The choice of the team form for all-gathers of one to two rounds, and the team form of the stack kernel on whole rounds (slices of 4 MiB and more), which it reads source by source: two
halves of four tiles, one partial result in LDS and one in registers.  Against the CPU checker, bit for bit."""
import numpy as np
import pytest

import closed_forms as cf
import gpu_harness as gh
from closed_forms import BF16, FP16, FP32, FP64, INT8, INT64, MAX, MIN, PROD, SUM

pytestmark = pytest.mark.gpu
H = gh.H
RING, RHD = 0, 2


@pytest.fixture(scope="module")
def orc():
    from oracle import oracle
    oracle.build()
    return oracle


# two and four servers, rounds of 8 and of 4 tiles, slices with a ragged end; max and min over NaNs and signed zeros, where a swapped operand changes the bits
@pytest.mark.parametrize("dt,op,p,servers,special,extra", [
    (FP32, MAX, 8, 2, True, 0), (FP32, MIN, 8, 4, True, 0), (FP32, SUM, 8, 2, False, 4099), (FP16, SUM, 8, 4, False, 0), (INT8, SUM, 8, 2, False, 0),
    (INT64, PROD, 9, 3, False, 0), (FP32, SUM, 10, 5, False, 0), (BF16, SUM, 8, 2, False, 0)])
def test_team_stack_whole_rounds(orc, dt, op, p, servers, special, extra):
    n = (p * (4 << 20) + extra) // H.DTYPE_SIZE[dt]
    rng = np.random.default_rng(9400 + dt + servers)
    pool = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1e-45, -1.0, 3.4e38], np.float32)
    plan = H.describe_plan(H.COLL_ALLREDUCE, RING | servers << 8, p, n, dt)
    assert {it["kind"] for it in plan["fused"]} == {3}
    print("team stack", dt, op, p, servers, special, extra, flush=True)
    ins = [rng.choice(pool, n).astype(np.float32) if special else cf.random_input(dt, n, rng) for _ in range(p)]
    want = orc.allreduce_two_level([x.copy() for x in ins], dt, op, servers, level1=RING)
    g = gh.Group(p, algo="ring", servers=servers, deterministic=1, team=1)
    try:
        for rep in range(2):
            outs, _ = gh.all_reduce(g, ins, dt, op)
            assert g.info()["teamLaunches"] >= 1
            for r in range(p):
                if special:
                    assert np.array_equal(outs[r].view(np.uint32), want[r].view(np.uint32)), r
                else:
                    assert gh.same(dt, outs[r], want[r]), r
    finally:
        g.close()


# 8-byte elements and 8-bit products: where more than a quarter of the tiles lie in items shorter than three quarters of a region (8 tiles for each
# of an XCD's 32 compute units) all are read tile by tile, else whole rounds source by source.  A slice goes in a third and two thirds.
@pytest.mark.parametrize("dt,op", [(INT64, SUM), (FP64, MAX), (INT8, PROD)])
@pytest.mark.parametrize("tiles,extra", [(95, 0), (191, 0), (192, 8), (257, 24)])
def test_team_stack_of_short_and_long_items(orc, dt, op, tiles, extra):
    p, servers = 8, 2
    n = p * 3 * (tiles * 16384 + extra) // H.DTYPE_SIZE[dt]
    plan = H.describe_plan(H.COLL_ALLREDUCE, RING | servers << 8, p, n, dt)
    assert {it["kind"] for it in plan["fused"]} == {3}
    print("team stack, short and long items", dt, op, tiles, extra, "items of", sorted({it["n"] for it in plan["fused"]}), flush=True)
    rng = np.random.default_rng(9700 + tiles + dt)
    ins = [cf.random_input(dt, n, rng) for _ in range(p)]
    want = orc.allreduce_two_level([x.copy() for x in ins], dt, op, servers, level1=RING)
    g = gh.Group(p, algo="ring", servers=servers, deterministic=1, team=1)
    try:
        for rep in range(2):
            outs, _ = gh.all_reduce(g, ins, dt, op)
            assert g.info()["teamLaunches"] >= 1
            for r in range(p):
                assert gh.same(dt, outs[r], want[r]), r
    finally:
        g.close()


@pytest.mark.parametrize("tiles,team", [(255, 0), (256, 1), (257, 1), (289, 1), (500, 1)])
def test_allgather_of_one_to_two_rounds(tiles, team):
    # `tiles` per rank; 8 x 256 tiles are a full round of 8 tiles on 256 compute units
    p, n = 8, tiles * 16384
    g = gh.Group(p)
    try:
        ins = [cf.random_input(INT8, n, np.random.default_rng(9600 + r)) for r in range(p)]
        print("all-gather, tiles per rank", tiles, flush=True)
        for rep in range(2):
            outs = gh.all_gather(g, ins, INT8)
            assert g.info()["teamLaunches"] == team
            whole = np.concatenate(ins)
            for r in range(p):
                assert np.array_equal(outs[r], whole), r
    finally:
        g.close()
