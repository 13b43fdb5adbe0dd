"""Chains of 8-bit elements whose blocks start off a word boundary: fetched as whole words and put together (kernels_impl.h,
WordVec); 16-bit ones beside them, which keep their 128-bit loads.  Reduce-scatter blocks of odd length start at every byte
offset; sizes around a vector, a pass and a tile, more sources than a batch holds; all-reduce in place with every rank's
buffer at another offset, where the words fetched hold bytes that neighbouring lanes write.  Against the CPU checker, bit for
bit, and the bytes around the buffers untouched."""
import numpy as np
import pytest
import torch

import closed_forms as cf
import gpu_harness as gh
from closed_forms import BF16, FP16, INT8, MAX, MIN, PROD, SUM, UINT8

pytestmark = pytest.mark.gpu
H = gh.H


@pytest.fixture(scope="module")
def orc():
    from oracle import oracle
    oracle.build()
    return oracle


@pytest.mark.parametrize("dt,op", [(INT8, SUM), (INT8, MAX), (INT8, PROD), (INT8, MIN), (UINT8, SUM), (UINT8, MAX), (FP16, SUM), (BF16, SUM)])
@pytest.mark.parametrize("p,pad", [(8, 0), (3, 2), (11, 0)])
def test_blocks_off_a_word_boundary(orc, dt, op, p, pad):
    g = gh.Group(p, algo="ring", team=0, direct=0)
    try:
        for n in (17, 255, 4097, 16383, 16401, 70001):
            print("word loads", dt, op, p, pad, n, flush=True)
            rng = np.random.default_rng(9500 + n + dt)
            ins = [cf.random_input(dt, n * p, rng) for _ in range(p)]
            want = orc.reducescatter(ins, dt, op)
            outs, keep = gh.reduce_scatter(g, ins, dt, op, pad=pad)
            assert g.info()["direct"] == 0 and g.info()["teamLaunches"] == 0
            for r in range(p):
                assert gh.same(dt, outs[r], want[r]), (n, r)
                assert np.array_equal(keep[r].view(np.uint8), ins[r].view(np.uint8))
    finally:
        g.close()


@pytest.mark.parametrize("dt,op", [(INT8, SUM), (INT8, MAX), (UINT8, PROD)])
@pytest.mark.parametrize("p,algo", [(4, "ring"), (9, "ring"), (6, "mesh")])
def test_in_place_at_every_offset(orc, dt, op, p, algo):
    g = gh.Group(p, algo=algo, team=0, direct=0)
    try:
        for n in (1, 16, 129 * p, 16384 * p + 5, 70001):
            print("word loads in place", dt, op, p, algo, n, flush=True)
            rng = np.random.default_rng(9550 + n + op)
            ins = [cf.random_input(dt, n, rng) for _ in range(p)]
            want = orc.allreduce(ins, dt, op, algo={"ring": 0, "mesh": 4 if op != PROD else 1}[algo])
            whole = [torch.full((n + 64,), 0xA5, dtype=torch.uint8, device="cuda") for _ in range(p)]
            bufs = [t[16 + 3 * r % 7:16 + 3 * r % 7 + n] for r, t in enumerate(whole)]
            for r in range(p):
                bufs[r].copy_(torch.from_numpy(ins[r].view(np.uint8)))
            torch.cuda.synchronize()
            ptrs = [t.data_ptr() for t in bufs]
            H.all_reduce(g.comms, ptrs, ptrs, n, dt, op, g.stream_ptr)
            g.stream.synchronize()
            assert g.info()["fused"] == 1 and g.info()["direct"] == 0 and g.info()["teamLaunches"] == 0
            for r in range(p):
                assert gh.same(dt, gh.to_host(bufs[r], dt), want[r]), (n, r)
                at = 16 + 3 * r % 7
                assert bool((whole[r][:at] == 0xA5).all()) and bool((whole[r][at + n:] == 0xA5).all()), (n, r)
    finally:
        g.close()
