"""Fused lists over general trees: allreduces on tori that are no powers of two, under AUTO.

CPU: a numpy model of the tree kernel (subtrees on a stack, then their join) gives the oracle's bits for the list that
AUTO runs, whose tree is never deeper than the kernel's stack.  GPU: oracle bits at the edges of tiles and vectors."""
import numpy as np
import pytest

from bine_trees_fugaku_amd import Batch, VComm
from bine_trees_fugaku_amd._lib import BineError
from bine_trees_fugaku_amd.collectives import plan_dump
from oracle import oracle as O
from tests import emulator as E
from tests.test_narrow import NP, data

TREE = 16
TORI = [[6], [10], [12], [6, 6], [2, 6, 2], [10, 10], [4, 6, 4]]


def stack_eval(values, pops):
    stack, deepest = [], 0
    for v, p in zip(values, pops):
        stack.append(v)
        deepest = max(deepest, len(stack))
        for _ in range(int(p)):
            b = stack.pop()
            stack[-1] = stack[-1] + b
    assert len(stack) == 1
    return stack[0], deepest


def run_trees(items, pool, bufs):
    def view(rb, off, n):
        return bufs[int(rb) >> 28][int(rb) & 0xFFFFFF, off:off + n]

    deepest = 0
    with np.errstate(over="ignore"):
        for it in items:
            assert it["flags"] == TREE and 1 <= it["lg"] <= 16
            n, d, at = int(it["n"]), int(it["delta"]), int(it["leaf_off"])
            cut = pool[at:at + int(it["lg"])]
            at += len(cut)
            sums = []
            for c in cut:
                leaves = pool[at:at + int(c["rb"])]
                at += -(-len(leaves) // 8) * 8
                v, depth = stack_eval([view(e["rb"], int(e["off"]) + d, n).copy() for e in leaves],
                                      (leaves["rb"] >> 24) & 15)
                deepest = max(deepest, depth)
                sums.append(v)
            total, depth = stack_eval(sums, cut["off"])
            deepest = max(deepest, depth)
            for e in pool[it["out_off"]:it["out_off"] + int(it["nouts"])]:
                view(e["rb"], int(e["off"]) + d, n)[...] = total
    return deepest


@pytest.mark.parametrize("dims", TORI)
@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("dtype", ["int8", "float32"])
def test_tree_lists(dims, in_place, dtype):
    P = int(np.prod(dims))
    for count in (P, 3 * P + 5, 330 * P + 1):
        if P * count > 3_000_000:
            continue
        x = data((P, count), dtype, count)
        meta, items, pool, launches = plan_dump(dims, "allreduce", count, dtype, in_place=in_place, exec="TREES")
        assert not meta["fused_ok"] and len(launches) == 1
        bufs = E.alloc_buffers(meta, NP[dtype], **({"recv": x} if in_place else {"send": x}))
        assert run_trees(items[::-1], pool, bufs) <= 12
        assert bufs[E.BUF_RECV].tobytes() == O.allreduce(x, dims).tobytes(), count


def test_rank_dependent_trees_stay_per_step():
    """Allreduce L on a ring of 130 builds many trees: fused it would move more than its steps do."""
    with pytest.raises(BineError):
        plan_dump([130], "allreduce", 130, "float32", exec="TREES", allreduce_algo="L")


@pytest.mark.gpu
@pytest.mark.parametrize("dims", TORI)
@pytest.mark.parametrize("dtype", ["int8", "int64", "float32"])
def test_trees_on_the_gpu(gpu, dims, dtype):
    import torch
    P = int(np.prod(dims))
    vec = 16 // np.dtype(NP[dtype]).itemsize
    with VComm(dims) as comm:
        for block in (1, vec, vec + 1, 64 * vec + 1, 129 * vec - 1):
            count = block * P + P // 2
            x = data((P, count), dtype, count)
            want = O.allreduce(x, dims).tobytes()
            s = torch.from_numpy(x).cuda()
            r = torch.zeros_like(s)
            comm.allreduce(s, r)
            comm.allreduce(s, s)
            torch.cuda.synchronize()
            assert r.cpu().numpy().tobytes() == want, block
            assert s.cpu().numpy().tobytes() == want, ("in place", block)
            s.copy_(torch.from_numpy(x))
            r.zero_()
            b = Batch(comm, [{"coll": "allreduce", "sendbuf": s, "recvbuf": r, "count": count}])
            b.launch_graph()
            torch.cuda.synchronize()
            assert r.cpu().numpy().tobytes() == want, ("batch", block)
            b.close()
