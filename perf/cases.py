"""Timed workloads of the framework, through its public entry points.

Every case is a dict of plain values.  The communicator (with its compiled schedule), the batch, the link simulation
or the network is what a program keeps between calls, so `prepare` builds it and issues one set-up call; `run` is one
pass with the buffers bound.  A torus is written "8x8x8"; `count` is the MPI count argument of the collective.

Kinds:
  allreduce   one allreduce; in_place: sendbuf is recvbuf (whole numbers only: the values are summed again each pass)
  shard       a reduce_scatter and the allgather of its result (a sharded optimizer's two collectives)
  alltoall    one alltoall, `count` elements per rank pair
  rooted      bcast, scatter, gather and reduce, root 0, of `count` elements per rank
  buckets     a batch of allreduces of uneven sizes, one work list
  linksim     one pass of the torus link simulation over whole tori, and every class's statistics
  selector    the selector's network: a forward pass over `queries` rows, loss and gradients of `batch` rows
"""
import math

import numpy as np
import torch

from bine_trees_fugaku_amd import Batch, VComm
from bine_trees_fugaku_amd import linksim as ls
from bine_trees_fugaku_amd import selector as sel

DTYPES = {"int8": torch.int8, "int32": torch.int32, "int64": torch.int64, "float32": torch.float32,
          "float64": torch.float64}


def _dims(case):
    return [int(d) for d in case["torus"].split("x")]


def _ranks(case):
    return math.prod(_dims(case))


def listed():
    return [
        # the smallest message: a few control words on eight ranks, where the call's own latency is the cost
        {"name": "allreduce_8_int32_4k", "kind": "allreduce", "torus": "2x2x2", "dtype": "int32", "count": 1024,
         "in_place": False},
        # a small layer's gradients on the largest torus: blocks of nine or ten elements, odd count
        {"name": "allreduce_512_fp32_odd", "kind": "allreduce", "torus": "8x8x8", "dtype": "float32", "count": 5003,
         "in_place": False},
        # MPI_IN_PLACE, 1 MiB per rank of the reference bench's INT32 type
        {"name": "allreduce_64_int32_inplace", "kind": "allreduce", "torus": "4x4x4", "dtype": "int32",
         "count": 262144, "in_place": True},
        # the largest: the headline allreduce, 4 MiB per rank on 512 ranks
        {"name": "allreduce_512_fp64_4m", "kind": "allreduce", "torus": "8x8x8", "dtype": "float64", "count": 524288,
         "in_place": False},
        # a torus that is no power of two, with the reference's validation count
        {"name": "allreduce_36_fp32", "kind": "allreduce", "torus": "6x6", "dtype": "float32", "count": 131072,
         "in_place": False},
        # bytes at an odd count: partitions and blocks at every alignment
        {"name": "allreduce_64_int8_odd", "kind": "allreduce", "torus": "4x4x4", "dtype": "int8", "count": 1048573,
         "in_place": False},
        # a sharded optimizer's step: reduce_scatter of the gradients, allgather of the parameters
        {"name": "shard_64_fp32", "kind": "shard", "torus": "4x4x4", "dtype": "float32", "count": 16411},
        # many small messages: 64 bytes for every pair of 512 ranks
        {"name": "alltoall_512_int32_64b", "kind": "alltoall", "torus": "8x8x8", "dtype": "int32", "count": 16},
        # the rooted collectives of a set-up or a metrics step: 16 KiB per rank on 512 ranks
        {"name": "rooted_512_fp32_16k", "kind": "rooted", "torus": "8x8x8", "dtype": "float32", "count": 4099},
        # gradient buckets of very different sizes in one batch
        {"name": "buckets_64_fp32", "kind": "buckets", "torus": "4x4x4", "dtype": "float32", "buckets": 32,
         "low": 4096, "high": 8388608, "layout": 7},
        # link traffic of every algorithm on five tori (the selector's held-out set)
        {"name": "linksim_5_tori", "kind": "linksim", "tori": "2x2x2 4x4x4 8x8x8 64x64 32x256"},
        # the selector's network at its training batch, and a ragged set of queries
        {"name": "selector_4096", "kind": "selector", "hidden": 256, "depth": 3, "batch": 4096, "queries": 1007},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["allreduce"] * 5 + ["shard", "alltoall", "rooted", "buckets", "linksim", "selector"])
    if kind == "linksim":
        n = rng.randint(2, 6)
        tori = ["x".join(map(str, t)) for t in rng.sample(sel.training_tori(max_p=8192), n)]
        return {"kind": kind, "tori": " ".join(tori)}
    if kind == "selector":
        return {"kind": kind, "hidden": rng.choice([128, 256]), "depth": rng.choice([2, 3]),
                "batch": _log_int(rng, 64, 8192), "queries": _log_int(rng, 1, 8192)}
    if kind == "buckets":
        return {"kind": kind, "torus": rng.choice(["2x2x2", "4x4", "4x8", "4x4x4"]),
                "dtype": rng.choice(["float32", "float64", "int32"]), "buckets": rng.randint(4, 40), "low": 4096,
                "high": _log_int(rng, 65536, 4194304), "layout": rng.randrange(1 << 20)}
    # one to eight gigabytes at most, 4 MiB per rank at most (per rank pair for alltoall: 16 KiB)
    if kind == "allreduce":
        in_place = rng.random() < 0.3
        torus = rng.choice(["2x2x2", "4x4", "4x8", "8x8", "4x4x4", "8x8x8", "6x6", "10x10", "4x6x4", "12"])
        dtype = rng.choice(["int8", "int32", "int64"] if in_place else ["int8", "int32", "int64", "float32", "float64"])
        case = {"kind": kind, "torus": torus, "dtype": dtype, "in_place": in_place}
        size = torch.empty((), dtype=DTYPES[dtype]).element_size()
        return {**case, "count": _log_int(rng, _ranks(case), (4 << 20) // size)}
    torus = rng.choice(["2x2x2", "4x4", "4x8", "8x8", "4x4x4", "8x8x8"])
    dtype = rng.choice(["int32", "int64", "float32", "float64"])
    case = {"kind": kind, "torus": torus, "dtype": dtype}
    size, ranks = torch.empty((), dtype=DTYPES[dtype]).element_size(), _ranks(case)
    most = {"shard": (4 << 20) // size // ranks, "alltoall": min((16 << 10) // size, (2 << 20) // size // ranks),
            "rooted": (1 << 20) // size}[kind]
    return {**case, "count": _log_int(rng, 1, most)}


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _values(shape, dtype, g):
    if dtype == torch.int8:
        return torch.randint(-128, 128, shape, dtype=dtype, device="cuda", generator=g)
    if not dtype.is_floating_point:
        return torch.randint(-1000, 1001, shape, dtype=dtype, device="cuda", generator=g)
    return torch.randn(shape, dtype=dtype, device="cuda", generator=g)


def _bucket_counts(case):
    rng = np.random.default_rng(case["layout"])
    size = torch.empty((), dtype=DTYPES[case["dtype"]]).element_size()
    b = np.exp(rng.uniform(math.log(case["low"]), math.log(case["high"]), case["buckets"]))
    return [max(1, int(x) // size) for x in b]


def _inputs(case, seed):
    """The input tensors of one state, from the seed alone."""
    g = _generator(seed)
    kind = case["kind"]
    if kind == "selector":
        dims = _net_dims(case)
        params = []
        for i, o in zip(dims[:-1], dims[1:]):
            params.append((torch.rand(o * i, device="cuda", generator=g) * 2 - 1) / math.sqrt(i))
            params.append((torch.rand(o, device="cuda", generator=g) * 2 - 1) * 0.1)
        n, q = case["batch"], case["queries"]
        x = torch.rand((n, dims[0]), device="cuda", generator=g)
        t = torch.randn((n, dims[-1]), device="cuda", generator=g)
        mask = (torch.rand((n, dims[-1]), device="cuda", generator=g) < 0.6).float()
        return {"params": torch.cat(params), "x": x, "t": t, "mask": mask,
                "q": torch.rand((q, dims[0]), device="cuda", generator=g)}
    if kind == "linksim":
        return {"sizes": torch.randint(8, 1 << 28, (26,), device="cuda", generator=g).cpu().numpy()}
    p, dt = _ranks(case), DTYPES[case["dtype"]]
    if kind == "buckets":
        return {"send": [_values((p, n), dt, g) for n in _bucket_counts(case)]}
    n = case["count"]
    if kind == "allreduce":
        return {"send": _values((p, n), dt, g)}
    if kind == "rooted":
        return {"bcast": _values((p, n), dt, g), "scatter": _values((p * n,), dt, g), "gather": _values((p, n), dt, g),
                "reduce": _values((p, n), dt, g)}
    return {"send": _values((p, p * n), dt, g)}  # shard, alltoall


def _net_dims(case):
    return [sel.N_FEATURES] + [case["hidden"]] * case["depth"] + [len(sel.OPTIONS)]


def _sim_cases(case):
    tori = [[int(d) for d in t.split("x")] for t in case["tori"].split()]
    return [(d, c, a) for d in tori for c, algos in ls.DEFINED.items() for a in algos
            if not (a == "simpy" and (len(set(d)) != 1 or d[0] > 1024))]  # its own range


def prepare(case, seed):
    s = _inputs(case, seed)
    s["kind"] = kind = case["kind"]
    if kind == "selector":
        s["net"] = sel.MLP(_net_dims(case), max_batch=8192)
        s["net"].set_params(s.pop("params").cpu().numpy())
        s["net"].forward(s["q"])
        return s
    if kind == "linksim":
        s["cases"] = len(_sim_cases(case))
        s["sim"] = ls.LinkSim(_sim_cases(case))
        s["sim"].run()
        return s
    comm = s["comm"] = VComm(_dims(case))
    if kind == "allreduce":
        s["recv"] = s["send"] if case["in_place"] else torch.empty_like(s["send"])
        # the set-up call compiles the schedule; in place it sums zeros, so the inputs stay as they are
        spare = torch.zeros_like(s["send"])
        comm.allreduce(spare, spare if case["in_place"] else s["recv"])
    elif kind == "shard":
        s["part"] = torch.empty((comm.size, case["count"]), dtype=s["send"].dtype, device="cuda")
        s["full"] = torch.empty_like(s["send"])
        run(s)
    elif kind == "alltoall":
        s["recv"] = torch.empty_like(s["send"])
        run(s)
    elif kind == "rooted":
        s["scattered"] = torch.empty_like(s["gather"])
        s["gathered"] = torch.empty_like(s["scatter"])
        s["reduced"] = torch.empty_like(s["reduce"][0])
        run(s)
    else:
        s["recv"] = [torch.empty_like(x) for x in s["send"]]
        s["batch"] = Batch(comm, [{"coll": "allreduce", "sendbuf": x, "recvbuf": y, "count": x.shape[1]}
                                  for x, y in zip(s["send"], s["recv"])])
        s["batch"].launch()
    return s


def run(s):
    kind = s["kind"]
    if kind == "allreduce":
        s["comm"].allreduce(s["send"], s["recv"])
        return s["recv"]
    if kind == "shard":
        s["comm"].reduce_scatter(s["send"], s["part"])
        s["comm"].allgather(s["part"], s["full"])
        return s["part"], s["full"]
    if kind == "alltoall":
        s["comm"].alltoall(s["send"], s["recv"])
        return s["recv"]
    if kind == "rooted":
        s["comm"].bcast(s["bcast"])
        s["comm"].scatter(s["scatter"], s["scattered"])
        s["comm"].gather(s["gather"], s["gathered"])
        s["comm"].reduce(s["reduce"], s["reduced"])
        return s["bcast"], s["scattered"], s["gathered"], s["reduced"]
    if kind == "buckets":
        s["batch"].launch()
        return s["recv"]
    if kind == "linksim":
        s["sim"].run()
        found = [s["sim"].stats(i) for i in range(s["cases"])]
        # every class's loads, and the bytes on its most loaded link at the state's message sizes
        mult, total, hops, num, den, rep = (np.concatenate([getattr(f, k) for f in found]).astype(np.int64)
                                            for k in ("max_mult", "sum_mult", "max_hops", "num", "den", "rep"))
        return {"mult": mult, "total": total, "hops": hops, "bytes": s["sizes"][:, None] * num // den * mult * rep}
    y = s["net"].forward(s["q"])
    loss, grads = s["net"].gradients(s["x"], s["t"], s["mask"])
    return y, loss, grads


def work(case):
    kind = case["kind"]
    if kind == "linksim":  # every class routes one message per rank (about ten operations) and fills its counters
        messages = counters = 0
        for d, c, a in _sim_cases(case):
            p = math.prod(d)
            n = len(ls.classes(d, c, a)["kind"])
            messages += n * p
            counters += n * p * len(d) * 2
        return {"bytes": 4 * counters, "flops": 10 * messages}
    if kind == "selector":
        dims = _net_dims(case)
        pairs = list(zip(dims[:-1], dims[1:]))
        macs = sum(i * o for i, o in pairs)
        back = 2 * macs - pairs[0][0] * pairs[0][1]  # no gradient of the inputs
        n, q = case["batch"], case["queries"]
        weights = macs + sum(dims[1:])
        io = n * (dims[0] + 2 * dims[-1]) + q * (dims[0] + dims[-1]) + 2 * weights
        return {"bytes": 4 * io, "flops": 2 * (q * macs + n * (macs + back))}
    p, size = _ranks(case), torch.empty((), dtype=DTYPES[case["dtype"]]).element_size()
    adds = 0
    if kind == "buckets":
        n = sum(_bucket_counts(case))
        elements, adds = 2 * p * n, (p - 1) * n
    elif kind == "allreduce":
        elements, adds = 2 * p * case["count"], (p - 1) * case["count"]
    elif kind == "shard":
        elements, adds = 2 * (p * p + p) * case["count"], (p - 1) * p * case["count"]
    elif kind == "alltoall":
        elements = 2 * p * p * case["count"]
    else:  # bcast and reduce: one partition against P; scatter and gather: P against P
        elements, adds = (2 * p + 4 * p) * case["count"], (p - 1) * case["count"]
    return {"bytes": elements * size, "flops": adds}


def _total(x):
    """Sum over the ranks: float64 for floating types, wrapping in its own type for whole numbers."""
    if x.dtype.is_floating_point:
        return x.double().sum(0)
    return x.sum(0, dtype=torch.int64).to(x.dtype)


def _everywhere(v, p):
    return v.expand(p, *v.shape).contiguous()


def exact(case, seed):
    kind = case["kind"]
    if kind == "linksim":
        return None  # whole numbers, equal or wrong
    s = _inputs(case, seed)
    if kind == "selector":
        dims = _net_dims(case)
        flat = s["params"].double()
        layers, at = [], 0
        for i, o in zip(dims[:-1], dims[1:]):
            w = flat[at:at + i * o].reshape(o, i)
            b = flat[at + i * o:at + i * o + o]
            layers.append((w, b))
            at += i * o + o

        def forward(x):
            acts = [x.double()]
            for k, (w, b) in enumerate(layers):
                z = acts[-1] @ w.t().contiguous() + b
                acts.append(z if k == len(layers) - 1 else z.clamp(min=0))
            return acts

        y = forward(s["q"])[-1]
        acts = forward(s["x"])
        m = s["mask"].double()
        d = (acts[-1] - s["t"].double()) * m
        count = m.sum().clamp(min=1)
        loss = (d * d).sum().reshape(1) / count
        dz, grads = 2 * d / count, []
        for k in range(len(layers) - 1, -1, -1):
            grads = [(dz.t().contiguous() @ acts[k]).reshape(-1), dz.sum(0)] + grads
            if k:
                dz = (dz @ layers[k][0]) * (acts[k] > 0)
        return y, loss, torch.cat(grads)
    p = _ranks(case)
    if kind == "allreduce":
        return _everywhere(_total(s["send"]), p)
    if kind == "buckets":
        return [_everywhere(_total(x), p) for x in s["send"]]
    n = case["count"]
    if kind == "alltoall":
        return s["send"].reshape(p, p, n).transpose(0, 1).reshape(p, p * n).contiguous()
    if kind == "shard":
        total = _total(s["send"])
        return total.reshape(p, n), _everywhere(total, p)
    return (_everywhere(s["bcast"][0], p), s["scatter"].reshape(p, n), s["gather"].reshape(p * n),
            _total(s["reduce"]))
