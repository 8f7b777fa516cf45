"""The launch shape a list starts with: one row per branch of the rule, by kind, size, fan and block length."""
import pytest

from bine_trees_fugaku_amd import Batch, VComm

GENERAL, GENERAL_STREAM, PAIR, BROAD = (1, 256, 0), (1, 256, 1), (2, 128, 1), (2, 256, 1)
QUAD, WIDE = (4, 128, 1), (4, 64, 1)

ROWS = [
    # below 64 MB, and lists that stay in the memory-side cache
    ("allreduce", [2, 2, 2], "int32", 262144, GENERAL), ("allreduce", [2, 4], "int32", 4194304, GENERAL),
    ("allreduce", [4, 4, 4], "float32", 507904, GENERAL), ("bcast", [16], "float32", 4194304, GENERAL),
    ("scatter", [2, 2, 2], "float32", 2097152, GENERAL), ("reduce_scatter", [2, 4], "float64", 262144, GENERAL),
    ("in place", [4, 4, 4], "int32", 262144, GENERAL), ("in place", [4, 4, 4], "float32", 1048576, GENERAL),
    ("reduce_scatter", [4, 4, 4], "float32", 16384, WIDE),
    # 64 to 96 MB, reductions out of place to 128 MB
    ("allreduce", [2, 4], "float32", 1310720, WIDE), ("allreduce", [16], "float32", 655360, QUAD),
    ("allreduce", [4, 8], "float32", 294912, PAIR), ("allreduce", [4, 4, 4], "float32", 163840, BROAD),
    ("allreduce", [4, 4, 4], "float32", 262144, BROAD), ("allreduce", [4, 4, 4], "float32", 266240, GENERAL),
    ("allreduce", [4, 4, 8], "float32", 79872, BROAD), ("allreduce", [4, 4, 8], "float32", 116736, GENERAL),
    ("allreduce", [4, 4, 4], "int8", 764925, GENERAL_STREAM), ("allreduce", [4, 4, 4], "int8", 1048573, PAIR),
    ("in place", [4, 4, 4], "int32", 163840, GENERAL),
    ("reduce_scatter", [16], "float32", 78080, QUAD), ("reduce_scatter", [4, 4, 4], "float32", 5120, PAIR),
    ("allgather", [4, 8], "float32", 17024, WIDE), ("alltoall", [4, 4, 4], "float32", 2560, GENERAL_STREAM),
    ("in place", [2, 4], "float32", 1310720, WIDE),
    # beyond the cache
    ("allreduce", [2, 4], "float32", 6291456, WIDE), ("allreduce", [4, 8], "int8", 6291456, WIDE),
    ("allreduce", [16, 16], "float32", 172032, BROAD), ("allreduce", [8, 8, 8], "float32", 83968, GENERAL_STREAM),
    ("allreduce", [4, 4, 4], "float32", 524288, QUAD), ("allreduce", [4, 4, 4], "int8", 2097152, GENERAL),
    ("allreduce", [4, 4, 4], "float32", 552957, QUAD), ("allreduce", [4, 4, 4], "int8", 2211837, GENERAL),
    ("allreduce", [4, 4, 4], "float32", 663552, QUAD), ("allreduce", [4, 4, 4], "float32", 819200, WIDE),
    ("allreduce", [4, 4, 8], "float32", 262144, GENERAL), ("allreduce", [4, 4, 8], "float32", 331776, PAIR),
    ("allreduce", [4, 4, 8], "float32", 655360, WIDE), ("allreduce", [4, 4, 8], "int8", 2621440, QUAD),
    ("allreduce", [16, 16], "int8", 1462272, PAIR), ("allreduce", [8, 8, 8], "float32", 139264, BROAD),
    ("allreduce", [8, 8, 8], "float32", 385024, QUAD),
    ("allreduce", [8, 8, 16], "float32", 45056, GENERAL), ("allreduce", [8, 8, 16], "float32", 65536, GENERAL),
    ("allreduce", [4, 4, 4], "float64", 1048576, WIDE), ("allgather", [16, 16], "float32", 1280, WIDE),
    ("bcast", [4, 4, 4], "float32", 1250048, GENERAL), ("bcast", [4, 4, 4], "float32", 1441792, WIDE),
    ("alltoall", [16, 16], "float32", 640, PAIR), ("in place", [4, 4, 4], "float32", 1835008, WIDE),
]


@pytest.mark.gpu
@pytest.mark.parametrize("coll,dims,dtype,count,shape", ROWS)
def test_starting_shape(gpu, coll, dims, dtype, count, shape):
    import torch
    t = getattr(torch, dtype)
    in_place = coll == "in place"
    coll = "allreduce" if in_place else coll
    with VComm(dims) as comm:
        P = comm.size
        n = {"allreduce": (P, P), "reduce_scatter": (P * P, P), "allgather": (P, P * P), "bcast": (0, P),
             "alltoall": (P * P, P * P), "scatter": (P, P)}[coll]
        r = torch.empty(n[1] * count, dtype=t, device="cuda")
        s = r if in_place else torch.empty(n[0] * count, dtype=t, device="cuda") if n[0] else None
        b = Batch(comm, [{"coll": coll, "sendbuf": s, "recvbuf": r, "count": count}])
        got = b.tuning()
        b.close()
    assert (got["vpt"], got["threads"], got["nontemporal"]) == shape


@pytest.mark.gpu
def test_many_small_buckets_start_with_the_narrow_kernel(gpu):
    """64-element blocks leave most lanes of a wider shape idle, whatever the list holds in all."""
    import torch
    with VComm([2, 2, 2]) as comm:
        count, n = 2048, 640
        s, r = (torch.empty(n, 8 * count, device="cuda") for _ in range(2))
        b = Batch(comm, [{"coll": "allreduce", "sendbuf": s[i], "recvbuf": r[i], "count": count} for i in range(n)])
        assert (b.tuning()["vpt"], b.tuning()["nontemporal"]) == (1, 0)
        b.close()
