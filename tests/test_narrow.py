"""The narrow lists of small calls (ITEM_NARROW): blocks shorter than a vector, vectors that overlap at a block's end,
trees and output lists spread over the lanes.

CPU: the narrow lowering of every schedule gives the oracle's bits under the host emulator, its items fit the kernel
and its blocks are covered once.  GPU: the kernel's bits equal the oracle's at the edges of its units and workgroups."""
import numpy as np
import pytest

from bine_trees_fugaku_amd import VComm
from bine_trees_fugaku_amd.collectives import plan_dump
from oracle import oracle as O
from tests import emulator as E

NP = {"int8": np.int8, "int32": np.int32, "int64": np.int64, "float32": np.float32, "float64": np.float64}
NARROW = 4
COLLS = ["allreduce", "reduce_scatter", "allgather", "bcast", "reduce"]


def data(shape, dtype, seed):
    rng = np.random.default_rng(seed)
    if dtype.startswith("int"):
        lim = np.iinfo(NP[dtype])
        return rng.integers(lim.min, lim.max, size=shape, endpoint=True).astype(NP[dtype])
    return (rng.standard_normal(shape) * 10.0 ** rng.uniform(-3, 3, shape)).astype(NP[dtype])


def inputs_and_result(coll, dims, dtype, count):
    """(sendbuf or None, recvbuf at the start or None, expected recvbuf)."""
    P = int(np.prod(dims))
    if coll == "allreduce":
        x = data((P, count), dtype, count)
        return x, None, O.allreduce(x, dims)
    if coll == "reduce_scatter":
        x = data((P, P * count), dtype, count)
        return x, None, O.reduce_scatter(x, dims)
    if coll == "allgather":
        x = data((P, count), dtype, count)
        return x, None, O.allgather(x, dims)
    if coll == "bcast":
        x = data((P, count), dtype, count)
        return None, x, np.broadcast_to(x[0], x.shape)
    x = data((P, count), dtype, count)
    return x, None, O.reduce(x, 0)


@pytest.mark.parametrize("coll", COLLS)
@pytest.mark.parametrize("dims", [[2], [2, 2, 2], [4, 4, 4]])
@pytest.mark.parametrize("dtype", ["int8", "int32", "float64"])
def test_narrow_lowering_matches_the_oracle(coll, dims, dtype):
    P = int(np.prod(dims))
    vec = 16 // np.dtype(NP[dtype]).itemsize
    for block in (1, vec - 1, vec, vec + 1, 4 * vec + 1, 65 * vec - 1):
        count = max(1, block if coll in ("reduce_scatter", "allgather") else block * P + P // 2)
        if P * P * count > 3_000_000:
            continue
        send, recv, want = inputs_and_result(coll, dims, dtype, count)
        meta, items, pool, launches = plan_dump(dims, coll, count, dtype, exec="FUSED", tile_elems=-1)
        assert (items["flags"] == NARROW).all() and len(launches) == 1
        bufs = E.alloc_buffers(meta, NP[dtype], send=send, recv=recv)
        E.run(meta, items, pool, launches, bufs)
        assert bufs[E.BUF_RECV].tobytes() == np.ascontiguousarray(want).tobytes(), (block, count)
        units = -(-items["n"].astype(int) // vec)
        assert (np.where(items["n"] >= vec, units, items["n"]) <= 1024).all()
        # every element of every output is written by one item
        wrote = sum(int(i["n"]) * int(i["nouts"]) for i in items)
        assert wrote == P * count * (P if coll == "allgather" else 1) - (count if coll == "bcast" else 0) \
            - ((P - 1) * count if coll == "reduce" else 0)


@pytest.mark.gpu
@pytest.mark.parametrize("coll", COLLS)
@pytest.mark.parametrize("dims", [[2, 2, 2], [4, 4, 4], [8, 8, 8]])
@pytest.mark.parametrize("dtype", ["int8", "int32", "int64", "float32", "float64"])
def test_narrow_kernel_matches_the_oracle(gpu, coll, dims, dtype):
    import torch
    P = int(np.prod(dims))
    vec = 16 // np.dtype(NP[dtype]).itemsize
    blocks = (1, vec + 1) if P == 512 else (1, vec - 1, vec, vec + 1, 4 * vec + 1, 65 * vec - 1)
    with VComm(dims, exec="FUSED") as comm:
        for block in blocks:
            count = max(1, block if coll in ("reduce_scatter", "allgather") else block * P + P // 2)
            if P * P * count > 6_000_000 and P < 512:
                continue
            send, recv, want = inputs_and_result(coll, dims, dtype, count)
            s = None if send is None else torch.from_numpy(send).cuda()
            r = torch.from_numpy(recv.copy()).cuda() if recv is not None else \
                torch.zeros(want.shape, dtype=s.dtype, device="cuda")
            getattr(comm, coll)(*([r] if s is None else [s, r]))
            torch.cuda.synchronize()
            assert r.cpu().numpy().tobytes() == np.ascontiguousarray(want).tobytes(), (block, count)
