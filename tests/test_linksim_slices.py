"""Link counts where a class's counters are held whole in a workgroup's LDS, one dimension at a time, or in memory."""
import numpy as np
import pytest

from bine_trees_fugaku_amd import linksim as ls
from oracle import oracle as O


@pytest.mark.gpu
@pytest.mark.parametrize("dims", [[2], [64], [16384], [128, 128], [16, 32, 32], [2, 8192], [65536], [256, 256]],
                         ids=lambda d: "x".join(map(str, d)))
def test_counts_by_size(gpu, dims):
    P = int(np.prod(dims))
    cases = [(dims, "allreduce", "recdoub"), (dims, "alltoall", "bine"), (dims, "bcast", "recdoub")]
    s = ls.LinkSim(cases + [([4, 4], "allreduce", "ring")])  # a small torus beside it
    for _ in range(2):
        s.run()
    for i, (d, coll, algo) in enumerate(s.cases):
        st = s.stats(i)
        n = len(st.num)
        for c in sorted({0, n // 2, n - 1}):
            dest = ls.peers(d, coll, algo, c).astype(np.int64)
            src = np.flatnonzero(dest != ls.NONE)
            want, longest = O.route_bytes(d, src, dest[src], 1)
            assert np.array_equal(s.link_counts(i, c), want.astype(np.uint32)), (coll, algo, c)
            assert (st.max_mult[c], st.sum_mult[c], st.max_hops[c]) == (want.max(), want.sum(), longest)
    s.close()
