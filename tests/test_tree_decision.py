"""Whether a schedule gets a list of general trees is told before the list is made, and only where some call may run it.

CPU: compiling a ring whose ranks each build a tree of their own (a list of 25 million leaves, which is not worth
running) takes the memory of its steps.  GPU: a communicator that was never AUTO compiles steps only; what it compiles
after it became AUTO runs as one launch, with the same bits."""
import subprocess
import sys

import pytest

from bine_trees_fugaku_amd import VComm
from oracle import oracle as O
from tests.conftest import ROOT
from tests.test_narrow import data

GROWTH = """
import resource, sys
from bine_trees_fugaku_amd._lib import BineError
from bine_trees_fugaku_amd.collectives import plan_dump
peak = lambda: resource.getrusage(resource.RUSAGE_SELF).ru_maxrss
plan_dump([6], "allreduce", 12, "float32", exec="STEP")
before = peak()
try:
    plan_dump([5000], "allreduce", 3, "float32", exec=sys.argv[1], allreduce_algo="L", in_place=sys.argv[2] == "1")
except BineError:
    assert sys.argv[1] == "TREES"
print((peak() - before) // 1024)
"""


@pytest.mark.parametrize("exec", ["STEP", "TREES"])
@pytest.mark.parametrize("in_place", ["0", "1"])
def test_refused_lists_are_not_made(exec, in_place):
    out = subprocess.run([sys.executable, "-c", GROWTH, exec, in_place], cwd=ROOT, capture_output=True, text=True)
    assert out.returncode == 0, out.stderr
    assert int(out.stdout) < 100, out.stdout  # MiB: the steps take 25, 25 million leaves of 8 bytes 190


@pytest.mark.gpu
def test_steps_alone_until_auto(gpu):
    import torch
    dims, P = [6, 6], 36
    with VComm(dims, exec="STEP") as comm:
        for count, launches in ((P + 5, "steps"), (2 * P + 1, "one"), (P + 5, "steps")):
            x = data((P, count), "float32", count)
            s = torch.from_numpy(x).cuda()
            r = torch.zeros_like(s)
            comm.allreduce(s, r)
            torch.cuda.synchronize()
            assert r.cpu().numpy().tobytes() == O.allreduce(x, dims).tobytes(), count
            n = comm.plan_stats("allreduce", count, "float32")["launches"]
            assert (n > 1) if launches == "steps" else (n == 1), (count, n)
            comm.set_exec("AUTO")
