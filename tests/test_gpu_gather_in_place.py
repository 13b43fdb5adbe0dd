"""All-gather in place (a rank's send buffer is its own block of its receive buffer): one fused pass that leaves that block
where it is, against the blocks themselves; small (descriptors in the kernel arguments), by tiles, in team form, with block
tables, over two servers, on some ranks only, and step by step (staged)."""
import numpy as np
import pytest
import torch

import gpu_harness as gh

pytestmark = pytest.mark.gpu
H = gh.H
INT8, BF16 = H.HCCL_DATA_TYPE_INT8, H.HCCL_DATA_TYPE_BFP16


@pytest.mark.parametrize("p,counts,servers,team,some", [
    (8, [1] * 8, 1, None, False), (8, [4099] * 8, 1, None, True), (16, [70001] * 16, 1, None, False), (8, [1300003] * 8, 1, None, False),
    (8, [1 << 20] * 8, 1, 1, True), (8, [12582912 + 3] * 8, 1, None, False), (8, [90001] * 8, 2, None, False),
    (4, [5, 400001, 17, 65536], 1, None, False), (4, [5, 400001, 17, 65536], 1, 1, True), (1, [1000], 1, None, False)])
def test_all_gather_in_place(p, counts, servers, team, some):
    for fuse in (1, 0):
        g = gh.Group(p, fuse=fuse, servers=servers, **({} if team is None else {"team": team}))
        try:
            for dt, pad in ((INT8, 3), (BF16, 16)):
                unit = H.DTYPE_SIZE[dt]
                print("all-gather in place", p, counts[0], "servers", servers, "team", team, "fuse", fuse, "type", dt, flush=True)
                gen = torch.Generator(device="cuda")
                gen.manual_seed(p + counts[0])
                displs = np.concatenate([[0], np.cumsum(counts)[:-1]])
                blocks = [torch.randint(0, 256, (n * unit,), dtype=torch.uint8, device="cuda", generator=gen) for n in counts]
                whole = [torch.full((sum(counts) * unit + pad + 64,), 0x5A, dtype=torch.uint8, device="cuda") for _ in range(p)]
                recvs = [t[pad:pad + sum(counts) * unit] for t in whole]
                sends = []
                for r in range(p):
                    if some and r % 3 == 1:
                        sends.append(blocks[r])
                        continue
                    mine = recvs[r][displs[r] * unit:(displs[r] + counts[r]) * unit]
                    mine.copy_(blocks[r])
                    sends.append(mine)
                torch.cuda.synchronize()
                want = torch.cat(blocks)
                for rep in range(2):
                    sp, rp = [t.data_ptr() for t in sends], [t.data_ptr() for t in recvs]
                    if len(set(counts)) > 1:
                        H.all_gather_v(g.comms, sp, rp, counts, displs, dt, g.stream_ptr)
                    else:
                        H.all_gather(g.comms, sp, rp, counts[0], dt, g.stream_ptr)
                    g.stream.synchronize()
                    info = g.info()
                    assert info["fused"] == fuse and (info["scratchBytes"] == 0 or fuse == 0), info
                    for r in range(p):
                        assert torch.equal(recvs[r], want), (dt, rep, r)
                        assert bool((whole[r][:pad] == 0x5A).all()) and bool((whole[r][pad + want.numel():] == 0x5A).all())
        finally:
            g.close()


def test_almost_in_place_is_staged():
    # one element beside its own block: the block would be overwritten while it is read
    p, n = 4, 3001
    g = gh.Group(p)
    try:
        recvs = [torch.zeros(n * p + 1, dtype=torch.int32, device="cuda") for _ in range(p)]
        blocks = [torch.arange(n, dtype=torch.int32, device="cuda") + 10000 * r for r in range(p)]
        sends = [recvs[r][r * n + 1:(r + 1) * n + 1] for r in range(p)]
        for s, b in zip(sends, blocks):
            s.copy_(b)
        torch.cuda.synchronize()
        H.all_gather(g.comms, [t.data_ptr() for t in sends], [t.data_ptr() for t in recvs], n, H.HCCL_DATA_TYPE_INT32, g.stream_ptr)
        g.stream.synchronize()
        assert g.info()["fused"] == 0
        for r in range(p):
            assert torch.equal(recvs[r][:n * p], torch.cat(blocks)), r
    finally:
        g.close()
