"""The tree kernel's deep instantiation: trees that need more than six values on the stack, as rings of some hundred
ranks and large tori do.

CPU: the lists need that depth, their waves take more than two groups of eight leaves, and the numpy model of the kernel
gives the oracle's bits.  GPU: the kernel's bits equal the oracle's, out of place, in place and in a captured batch."""
import numpy as np
import pytest

from bine_trees_fugaku_amd import Batch, VComm
from bine_trees_fugaku_amd.collectives import plan_dump
from oracle import oracle as O
from tests import emulator as E
from tests.test_narrow import NP, data
from tests.test_trees import run_trees

CASES = [([400], "B"), ([12, 12, 6], "L"), ([1000], "B")]


def longest(items, pool):
    return max(int(e["rb"]) for it in items for e in pool[it["leaf_off"]:it["leaf_off"] + it["lg"]])


@pytest.mark.parametrize("dims,algo", CASES)
@pytest.mark.parametrize("in_place", [False, True])
def test_lists_need_the_deep_stack(dims, algo, in_place):
    P = int(np.prod(dims))
    if in_place and P > 400:
        pytest.skip("L in place runs per step; B is compiled out of place")
    count = 16389 if algo == "L" else P + 5
    x = data((P, count), "float32", count)
    meta, items, pool, _ = plan_dump(dims, "allreduce", count, "float32", in_place=in_place, exec="TREES",
                                     allreduce_algo=algo)
    bufs = E.alloc_buffers(meta, NP["float32"], **({"recv": x} if in_place else {"send": x}))
    assert 6 < run_trees(items, pool, bufs) <= 12
    assert longest(items, pool) > 16
    assert bufs[E.BUF_RECV].tobytes() == O.allreduce(x, dims, algo=algo).tobytes()


@pytest.mark.gpu
@pytest.mark.parametrize("dims,algo", CASES)
@pytest.mark.parametrize("dtype", ["int8", "int64", "float32", "float64"])
def test_deep_stack_on_the_gpu(gpu, dims, algo, dtype):
    import torch
    P = int(np.prod(dims))
    vec = 16 // np.dtype(NP[dtype]).itemsize
    counts = [4096 * vec + 5] if algo == "L" else [P + P // 2, (vec + 1) * P + 7]
    if P == 1000:
        if dtype != "float32":
            pytest.skip("compiled for one type")
        counts = counts[:1]
    with VComm(dims, allreduce_algo=algo) as comm:
        for count in counts:
            x = data((P, count), dtype, count)
            want = O.allreduce(x, dims, algo=algo).tobytes()
            s = torch.from_numpy(x).cuda()
            r = torch.zeros_like(s)
            comm.allreduce(s, r)
            comm.allreduce(s, s)
            torch.cuda.synchronize()
            assert r.cpu().numpy().tobytes() == want, count
            assert s.cpu().numpy().tobytes() == want, ("in place", count)
            assert comm.plan_stats("allreduce", count, dtype)["launches"] == 1
            s.copy_(torch.from_numpy(x))
            r.zero_()
            b = Batch(comm, [{"coll": "allreduce", "sendbuf": s, "recvbuf": r, "count": count}])
            b.launch_graph()
            torch.cuda.synchronize()
            assert r.cpu().numpy().tobytes() == want, ("batch", count)
            b.close()
