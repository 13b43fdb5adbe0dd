"""Chains of 8- and 16-bit elements whose blocks start off a word boundary: fetched as whole words and put together
(kernels_impl.h, WordVec).  Reduce-scatter blocks of odd length start at every byte offset; sizes around a vector, a pass
and a tile, more sources than a batch holds; against the CPU checker, bit for bit."""
import numpy as np
import pytest

import closed_forms as cf
import gpu_harness as gh
from closed_forms import BF16, FP16, INT8, MAX, PROD, SUM

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def orc():
    from oracle import oracle
    oracle.build()
    return oracle


@pytest.mark.parametrize("dt,op", [(INT8, SUM), (INT8, MAX), (FP16, SUM), (BF16, SUM), (BF16, PROD), (BF16, MAX)])
@pytest.mark.parametrize("p,pad", [(8, 0), (3, 2), (11, 0)])
def test_blocks_off_a_word_boundary(orc, dt, op, p, pad):
    # blocks_per_cu = 1: the tile kernels also for sizes the argument-borne launch would take
    g = gh.Group(p, algo="ring", team=0, blocks_per_cu=1)
    try:
        for n in (17, 255, 4097, 16383, 16401, 70001):
            print("word loads", dt, op, p, pad, n, flush=True)
            rng = np.random.default_rng(9500 + n + dt)
            ins = [cf.random_input(dt, n * p, rng) for _ in range(p)]
            want = orc.reducescatter(ins, dt, op)
            outs, keep = gh.reduce_scatter(g, ins, dt, op, pad=pad)
            for r in range(p):
                assert gh.same(dt, outs[r], want[r]), (n, r)
                assert np.array_equal(keep[r].view(np.uint8), ins[r].view(np.uint8))
    finally:
        g.close()
