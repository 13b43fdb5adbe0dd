"""All-to-all-v called again: the same tables, one count moved, only displacements moved, other buffers, another
collective in between, a call that is refused -- every call moves what its own tables say."""
import numpy as np
import pytest
import torch

import gpu_harness as gh

pytestmark = pytest.mark.gpu
H = gh.H


def _tables(rng, p, hi):
    cnt = rng.integers(0, hi, (p, p)).astype(np.uint64)
    before = lambda c: np.cumsum(c, axis=1, dtype=np.uint64) - c  # noqa: E731
    return cnt, before(cnt), np.ascontiguousarray(cnt.T), before(np.ascontiguousarray(cnt.T))


def _want(p, sends, t, room):
    cnt, sd, back, rd = (x.astype(np.int64) for x in t)
    outs = [np.full(room, -1, np.int32) for _ in range(p)]
    for i in range(p):
        for j in range(p):
            outs[j][rd[j, i]:rd[j, i] + cnt[i, j]] = sends[i][sd[i, j]:sd[i, j] + cnt[i, j]]
    return outs


@pytest.mark.parametrize("p,hi", [(4, 700), (64, 60), (9, 9000)])
def test_repeated_and_changed_tables(p, hi):
    g = gh.Group(p)
    try:
        rng = np.random.default_rng(9700 + p)
        room = p * hi * 2
        sends = [[rng.integers(-(1 << 30), 1 << 30, room).astype(np.int32) for _ in range(p)] for _ in range(2)]
        dev = [[gh.to_dev(x) for x in s] for s in sends]
        out = [torch.empty(room, dtype=torch.int32, device="cuda") for _ in range(p)]

        def call(t, k, expect_hit=None):
            for o in out:
                o.fill_(-1)
            torch.cuda.synchronize()
            H.all_to_all_v(g.comms, [x.data_ptr() for x in dev[k]], t[0], t[1], [x.data_ptr() for x in out], t[2], t[3], H.HCCL_DATA_TYPE_INT32, g.stream_ptr)
            g.stream.synchronize()
            if expect_hit is not None:
                assert g.info()["cacheHit"] == expect_hit
            for r, w in enumerate(_want(p, sends[k], t, room)):
                assert np.array_equal(out[r].cpu().numpy(), w), r

        a, b = _tables(rng, p, hi), _tables(rng, p, hi)
        call(a, 0, 0)
        call(a, 0, 1)
        call(a, 1, 0)                                     # other buffers
        call(a, 1, 1)
        call(a, 0, 1)                                     # the first ones again
        call(b, 0, 0)
        call(a, 0, 1)
        call(a, 0, 1)
        moved = [x.copy() for x in a]                     # one pair exchanges one element less
        i, j = np.argwhere(a[0] > 0)[-1]
        moved[0][i, j] -= 1
        moved[2][j, i] -= 1
        call(moved, 0, 0)
        call(moved, 0, 1)
        shifted = [x.copy() for x in moved]               # only displacements differ
        shifted[3][p - 1] += np.uint64(3)
        call(shifted, 0, 0)
        call(shifted, 0, 1)
        x = [torch.ones(1000, dtype=torch.float32, device="cuda") for _ in range(p)]
        torch.cuda.synchronize()
        H.all_reduce(g.comms, [t.data_ptr() for t in x], [t.data_ptr() for t in x], 1000, H.HCCL_DATA_TYPE_FP32, H.HCCL_REDUCE_SUM, g.stream_ptr)
        call(shifted, 0, 1)
        bad = [t.copy() for t in shifted]                 # rank 0 expects more than is sent: refused, and forgotten
        bad[2][0, p - 1] += np.uint64(1)
        with pytest.raises(H.HcclError):
            call(bad, 0)
        with pytest.raises(H.HcclError):
            call(bad, 0)
        call(shifted, 0, 1)
        H.set_param(g.comms[0], "fuse", 0)                # a setting is part of what was prepared
        call(shifted, 0, 0)
        call(shifted, 0, 1)
        H.set_param(g.comms[0], "fuse", 1)
        call(shifted, 0, 1)
    finally:
        g.close()
