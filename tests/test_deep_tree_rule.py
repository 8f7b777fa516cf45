"""Which lists of deep general trees AUTO runs: where few blocks hold very many leaves each, the schedule's steps are
faster at small counts, and at any count where they move no more than the list."""
import pytest

from bine_trees_fugaku_amd._lib import BineError
from bine_trees_fugaku_amd.collectives import plan_dump


@pytest.mark.parametrize("dims,algo,count,dtype,listed", [
    ([20, 20], "L", 3, "float32", False), ([20, 20], "L", 1000, "float32", False),
    ([20, 20], "L", 8192, "float32", True), ([20, 20], "L", 65536, "float32", False),
    ([12, 12, 6], "L", 1000, "float32", False), ([12, 12, 6], "L", 65536, "float32", True),
    ([10, 10, 10], "L", 1000, "float32", False), ([10, 10, 10], "L", 20000, "float64", True),
    ([18, 18], "L", 3, "float32", True), ([400], "B", 403, "float32", True), ([400], "B", 131072, "int8", True),
    ([24, 24], "B", 600, "float64", True)])
def test_deep_lists(dims, algo, count, dtype, listed):
    def dump():
        return plan_dump(dims, "allreduce", count, dtype, exec="TREES", allreduce_algo=algo)
    if listed:
        assert len(dump()[3]) == 1
    else:
        with pytest.raises(BineError):
            dump()
