"""Grids of short copies (ITEM_PACK): alltoall, scatter and gather of short and odd blocks.

CPU: the grids expand to every copy of the collective once, with the oracle's result, in fused and per-step lists.
GPU: results at block lengths around the kernel's units, for every element type."""
import numpy as np
import pytest

from bine_trees_fugaku_amd import Batch, VComm
from bine_trees_fugaku_amd.collectives import plan_dump
from oracle import oracle as O
from tests import emulator as E
from tests.test_narrow import NP, data

PACK = 32
M32 = 0xFFFFFFFF


def expand(items, pool):
    """The launch's grids as ordinary one-copy items."""
    out_items, out_pool = [], list(pool)
    for it in items:
        if it["flags"] != PACK:
            out_items.append(it)
            continue
        l0, o0, l1, o1, l2, o2 = ([int(v) for v in e] for e in pool[it["leaf_off"]:it["leaf_off"] + 6])
        for j2 in range(int(it["pad"]) >> 16):
            for j1 in range(int(it["pad"]) & 0xFFFF):
                one = it.copy()
                one["flags"], one["pad"], one["nouts"], one["lg"] = 0, 0, 1, 0
                one["leaf_off"], one["out_off"] = len(out_pool), len(out_pool) + 1
                for a, b, c in ((l0, l1, l2), (o0, o1, o2)):
                    out_pool.append(tuple((a[i] + b[i] * j1 + c[i] * j2) & M32 for i in range(2)))
                out_items.append(one)
    return np.array(out_items, items.dtype), np.array([tuple(e) for e in out_pool], pool.dtype)


def case(coll, P, dtype, count):
    """(sendbuf, expected recvbuf) of a copy collective."""
    if coll == "alltoall":
        x = data((P, P * count), dtype, count)
        return x, O.alltoall(x, P)
    if coll == "scatter":
        x = data((P * count,), dtype, count)
        return x, x.reshape(P, count)
    x = data((P, count), dtype, count)
    return x, x.reshape(-1)


@pytest.mark.parametrize("coll", ["alltoall", "scatter", "gather"])
@pytest.mark.parametrize("P", [2, 8, 32])
@pytest.mark.parametrize("exec", ["FUSED", "STEP"])
@pytest.mark.parametrize("kw", [{}, {"alltoall_family": "BRUCK"}])
def test_grids_hold_every_copy(coll, P, exec, kw):
    if kw and coll != "alltoall":
        pytest.skip("an alltoall family")
    for dtype, count in (("int8", 3), ("int8", 40), ("int32", 1), ("int32", 131), ("float64", 199)):
        send, want = case(coll, P, dtype, count)
        meta, items, pool, launches = plan_dump([P], coll, count, dtype, exec=exec, tile_elems=-4096, **kw)
        assert (items["flags"] == PACK).any()
        bufs = E.alloc_buffers(meta, NP[dtype], send=send)
        written = 0
        for first, n in launches:
            its, pl = expand(items[first:first + n], pool)
            E.run(meta, its, pl, [(0, len(its))], bufs, reverse=True)
            written += sum(int(i["n"]) * int(i["nouts"]) for i in its)
        assert bufs[E.BUF_RECV].reshape(np.shape(want)).tobytes() == np.ascontiguousarray(want).tobytes(), (dtype, count)
        if exec == "FUSED":
            assert written == np.size(want)


@pytest.mark.gpu
@pytest.mark.parametrize("coll", ["alltoall", "scatter", "gather"])
@pytest.mark.parametrize("P", [8, 64])
@pytest.mark.parametrize("dtype", ["int8", "int32", "int64", "float32", "float64"])
def test_packs_on_the_gpu(gpu, coll, P, dtype):
    import torch
    size = np.dtype(NP[dtype]).itemsize
    with VComm([P]) as comm:
        for nbytes in (size, 3 * size, 7 * size, 16, 17 * size, 2048, 2048 + size, 20480 - size, 20480 + size):
            if P == 64 and coll == "alltoall" and nbytes > 3000:
                continue
            count = nbytes // size
            send, want = case(coll, P, dtype, count)
            s = torch.from_numpy(np.ascontiguousarray(send)).cuda()
            r = torch.zeros(np.shape(want), dtype=s.dtype, device="cuda")
            getattr(comm, coll)(s, r)
            torch.cuda.synchronize()
            assert r.cpu().numpy().tobytes() == np.ascontiguousarray(want).tobytes(), count
            r.zero_()
            b = Batch(comm, [{"coll": coll, "sendbuf": s, "recvbuf": r, "count": count}])
            b.launch()
            torch.cuda.synchronize()
            assert r.cpu().numpy().tobytes() == np.ascontiguousarray(want).tobytes(), ("batch", count)
            b.close()
