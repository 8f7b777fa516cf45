"""Autotuning where a list of general trees runs: no launch shape changes such a list, so none is chosen for it."""
import numpy as np
import pytest

from bine_trees_fugaku_amd import Batch, VComm
from bine_trees_fugaku_amd._lib import BineError
from oracle import oracle as O
from tests.test_narrow import data


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [[6], [6, 6]])
def test_tree_lists_keep_their_shape(gpu, dims):
    import torch
    P = int(np.prod(dims))
    count = 100 * P + 3
    x = data((P, count), "float32", count)
    want = O.allreduce(x, dims).tobytes()
    s = torch.from_numpy(x).cuda()
    r = torch.zeros_like(s)
    with VComm(dims, alltoall_family="BRUCK") as comm:
        b = Batch(comm, [{"coll": "allreduce", "sendbuf": s, "recvbuf": r, "count": count}])
        start = b.tuning()
        b.autotune(iters=1)
        assert b.tuning() == start
        b.launch_graph()
        torch.cuda.synchronize()
        assert r.cpu().numpy().tobytes() == want
        b.close()
        r.zero_()
        comm.autotune("allreduce", s, r, count, iters=1)
        torch.cuda.synchronize()
        assert r.cpu().numpy().tobytes() == want
        with pytest.raises(BineError):  # buffers are checked all the same
            comm.autotune("allreduce", s, torch.zeros(P, device="cuda"), 1 << 20, iters=1)
        # an ordinary list beside the trees is tuned
        a = data((P, P * 8), "float32", 8)
        p = torch.from_numpy(a).cuda()
        q = torch.zeros_like(p)
        b = Batch(comm, [{"coll": "allreduce", "sendbuf": s, "recvbuf": r, "count": count},
                         {"coll": "alltoall", "sendbuf": p, "recvbuf": q, "count": 8}])
        r.zero_()
        b.autotune(iters=1)
        b.launch()
        torch.cuda.synchronize()
        assert r.cpu().numpy().tobytes() == want
        assert q.cpu().numpy().tobytes() == a.reshape(P, P, 8).transpose(1, 0, 2).tobytes()
        b.close()
