"""Vector items whose first and last vectors overlap their neighbours (blocks of any length at any alignment).

CPU: the lowering gives the oracle's bits under the host emulator, its items share no output, and the vectors the
kernel derives from an item cover exactly the item.  GPU: oracle bits at several launch shapes, blocks one element
around the tile lengths, element types down to bytes at odd counts."""
import numpy as np
import pytest

from bine_trees_fugaku_amd import Batch, VComm
from bine_trees_fugaku_amd.collectives import plan_dump
from oracle import oracle as O
from tests import emulator as E
from tests.test_narrow import COLLS, NP, inputs_and_result

VECTOR, RUN = 1 | 8, 2


@pytest.mark.parametrize("coll", COLLS)
@pytest.mark.parametrize("dims", [[2, 2], [2, 2, 2]])
@pytest.mark.parametrize("dtype", ["int8", "float32", "float64"])
@pytest.mark.parametrize("two_phase", [0, 1, 2, 5])
def test_shared_ends_lowering(coll, dims, dtype, two_phase):
    P = int(np.prod(dims))
    vec = 16 // np.dtype(NP[dtype]).itemsize
    tile = 16 * vec
    for block in (1, vec - 1, vec, vec + 1, tile - 1, tile, tile + 1, tile + vec - 1, 2 * tile + 1, 5 * tile + 3):
        count = max(1, block if coll in ("reduce_scatter", "allgather") else block * P + P // 2)
        send, recv, want = inputs_and_result(coll, dims, dtype, count)
        meta, items, pool, launches = plan_dump(dims, coll, count, dtype, exec="FUSED", tile_elems=-tile,
                                                two_phase=two_phase)
        bufs = E.alloc_buffers(meta, NP[dtype], send=send, recv=recv)
        E.run(meta, items, pool, launches, bufs, reverse=True)
        assert bufs[E.BUF_RECV].tobytes() == np.ascontiguousarray(want).tobytes(), (block, count)
        for first, n in launches:  # no two items of a launch write one element
            seen = {}
            for it in items[first:first + n]:
                if it["flags"] & RUN:
                    continue
                for e in pool[it["out_off"]:it["out_off"] + it["nouts"]]:
                    lo = int(e["off"]) + int(it["delta"])
                    seen.setdefault(int(e["rb"]), []).append((lo, lo + int(it["n"])))
            for spans in seen.values():
                spans.sort()
                assert all(a[1] <= b[0] for a, b in zip(spans, spans[1:]))
        for it in items:
            if not it["flags"] & VECTOR or it["flags"] & RUN:
                continue
            n, pad = int(it["n"]), int(it["pad"])
            assert n >= vec and pad < vec and n <= (2 if two_phase & 4 else 1) * tile
            starts = np.clip(np.arange(-(-(n + pad) // vec)) * vec - pad, 0, n - vec)
            covered = np.zeros(n, bool)
            for s in starts:
                covered[s:s + vec] = True
            assert covered.all()


@pytest.mark.gpu
@pytest.mark.parametrize("coll", COLLS)
@pytest.mark.parametrize("dtype", ["int8", "int32", "float64"])
def test_blocks_around_the_tile_lengths(gpu, coll, dtype):
    import torch
    dims, P = [4, 4, 4], 64
    vec = 16 // np.dtype(NP[dtype]).itemsize
    with VComm(dims, exec="FUSED") as comm:
        for block in (vec + 1, 64 * vec - 1, 256 * vec + 1, 300 * vec + vec - 1):
            count = block if coll in ("reduce_scatter", "allgather") else block * P + 5
            send, recv, want = inputs_and_result(coll, dims, dtype, count)
            s = None if send is None else torch.from_numpy(send).cuda()
            start = recv if recv is not None else np.zeros(want.shape, NP[dtype])
            r = torch.from_numpy(start.copy()).cuda()
            b = Batch(comm, [{"coll": coll, "sendbuf": s, "recvbuf": r, "count": count}])
            for vpt, threads, nt, two_phase in [(1, 256, 0, 0), (4, 64, 1, 0), (2, 512, 0, 2), (1, 128, 1, 1)]:
                r.copy_(torch.from_numpy(start))
                b.set_tuning(vpt, threads, 0, nt, two_phase=two_phase)
                b.launch()
                torch.cuda.synchronize()
                got = r.cpu().numpy()
                assert got.tobytes() == np.ascontiguousarray(want).tobytes(), (block, vpt, threads, two_phase)
            b.close()
