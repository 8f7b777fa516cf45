"""Which short blocks of an allreduce the narrow kernel takes: fewer units the more leaves they have, and more of them
where blocks are whole lines in a list beyond the memory-side cache.  The general shape's tiles are 64 units there."""
import pytest

from bine_trees_fugaku_amd import VComm


@pytest.mark.gpu
@pytest.mark.parametrize("dims,count,narrow", [
    ([16, 16], 49152, True), ([16, 16], 65536, True), ([16, 16], 81920, False), ([16, 16], 98496, False),
    ([8, 8, 8], 65920, True), ([16, 8, 8], 66304, True), ([16, 8, 8], 131072, True)])
def test_short_blocks(gpu, dims, count, narrow):
    with VComm(dims) as comm:
        P = comm.size
        block = -(-count // P)
        general = P * (-(-block // 256))
        items = comm.plan_stats("allreduce", count, "float32")["items"]
        assert (items != general) if narrow else (items == general), (items, general)
