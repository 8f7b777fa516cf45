"""In-place allreduces as fused lists: each work item reads its elements of every rank before it writes any.

CPU: the list AUTO runs, in every lowering and item order, gives the oracle's bits, and a schedule whose groups read
what another group writes stays per step.  GPU: oracle bits for each kernel path (narrow, split trees, shallow trees,
one-wave workgroups, two phases) at odd counts, single calls and batches."""
import numpy as np
import pytest

from bine_trees_fugaku_amd import Batch, VComm
from bine_trees_fugaku_amd.collectives import plan_dump
from oracle import oracle as O
from tests import emulator as E
from tests.test_narrow import NP, data
from tests.test_packs import expand

VECTOR = 1 | 8


@pytest.mark.parametrize("dims", [[2], [8], [4, 4], [2, 2, 2], [4, 4, 4]])
@pytest.mark.parametrize("algo", ["B", "B_CONT", "B_COALESCE", "L"])
@pytest.mark.parametrize("tile,two_phase", [(16, 0), (16, 1), (-1, 0), (-64, 0), (-64, 2), (-64, 5)])
def test_in_place_lists(dims, algo, tile, two_phase):
    P = int(np.prod(dims))
    for count in (P, 7 * P + 3, 70 * P + 1):
        x = data((P, count), "float32", count)
        kw = dict(in_place=True, allreduce_algo=algo, exec="AUTO", tile_elems=tile, two_phase=two_phase)
        meta, items, pool, launches = plan_dump(dims, "allreduce", count, "float32", **kw)
        assert not meta["fused_ok"]  # exec = FUSED refuses an in-place call, as ever
        if algo == "B":
            assert len(launches) == (1 if two_phase == 0 or tile == -1 else 2)
        for reverse in (False, True):
            bufs = E.alloc_buffers(meta, np.float32, recv=x)
            for first, n in launches:  # per-step lists (algorithm L) may hold grids of copies
                its, pl = expand(items[first:first + n], pool)
                E.run(meta, its, pl, [(0, len(its))], bufs, reverse=reverse)
            want = O.allreduce(x, dims, algo=algo)
            assert bufs[E.BUF_RECV].tobytes() == want.tobytes(), (count, reverse)


def test_ranks_with_different_trees_stay_per_step():
    """Algorithm L on a ring of 8 leaves rank-dependent trees: one group's outputs are another's leaves."""
    meta, items, pool, launches = plan_dump([8], "allreduce", 64, "float64", in_place=True, allreduce_algo="L",
                                            exec="AUTO")
    assert len(launches) > 1 and (items["lg"] <= 1).all()


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [[2, 2, 2], [4, 4], [4, 4, 4], [8, 8, 8]])
@pytest.mark.parametrize("dtype", ["int8", "float32", "float64"])
def test_in_place_on_the_gpu(gpu, dims, dtype):
    import torch
    P = int(np.prod(dims))
    vec = 16 // np.dtype(NP[dtype]).itemsize
    for block in ((vec + 1, 129 * vec + 1) if P < 512 else (2,)) + ((1100 * vec + 3,) if P <= 16 else ()):
        count = block * P + P // 2 + 1
        x = data((P, count), dtype, count)
        want = O.allreduce(x, dims)
        buf = torch.from_numpy(x).cuda()
        with VComm(dims) as comm:
            comm.allreduce(buf, buf)
            torch.cuda.synchronize()
            assert buf.cpu().numpy().tobytes() == want.tobytes(), block
            b = Batch(comm, [{"coll": "allreduce", "sendbuf": buf, "recvbuf": buf, "count": count}])
            for vpt, threads, nt, two_phase, double in [(1, 256, 0, 0, 0), (4, 64, 1, 0, 0), (2, 512, 0, 0, 0),
                                                        (1, 128, 1, 1, 0), (4, 64, 1, 2, 1), (1, 256, 1, 0, 0)]:
                buf.copy_(torch.from_numpy(x))
                b.set_tuning(vpt, threads, 0, nt, two_phase=two_phase, double_tiles=double)
                b.launch()
                torch.cuda.synchronize()
                assert buf.cpu().numpy().tobytes() == want.tobytes(), (block, vpt, threads, two_phase)
            b.close()
