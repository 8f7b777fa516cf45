"""The pack kernel is a launch of its own: beside other items it only runs where thousands of short copies pay for it."""
import numpy as np
import pytest

from bine_trees_fugaku_amd.collectives import plan_dump
from oracle import oracle as O
from tests import emulator as E
from tests.test_narrow import data
from tests.test_packs import PACK, expand


@pytest.mark.parametrize("dims,count,dtype", [([6, 6], 131072, "float32"), ([4, 4, 4], 65547, "float32"),
                                              ([2, 2, 2], 20011, "float32"), ([8, 8], 100003, "int8"),
                                              ([4, 4, 4], 16384, "float32")])
def test_packs_add_no_launch_to_a_step(dims, count, dtype):
    P = int(np.prod(dims))
    x = data((P, count), dtype, count)
    meta, items, pool, launches = plan_dump(dims, "allreduce", count, dtype, exec="STEP", tile_elems=-1024)
    bufs = E.alloc_buffers(meta, x.dtype.type, send=x)
    for first, n in launches:
        packs = items["flags"][first:first + n] == PACK
        assert packs.all() or not packs.any(), (packs.sum(), n)
        its, pl = expand(items[first:first + n], pool)
        E.run(meta, its, pl, [(0, len(its))], bufs)
    assert bufs[E.BUF_RECV].tobytes() == O.allreduce(x, dims).tobytes()


def test_many_short_copies_are_packed_beside_others():
    # an allgather's steps on 512 ranks forward thousands of short blocks, some of them in runs of longer ones
    _, items, _, launches = plan_dump([8, 8, 8], "allreduce", 512 * 32 + 7, "float32", exec="STEP", tile_elems=-1024)
    assert (items["flags"] == PACK).any()
