"""The work that programs have this partitioner do, as cases to be timed.

A case is one call (or one batch of calls) through the public entry points on
a graph of one of the kinds the configurations, tests and benchmark use:

* ``mesh``   -- a 2-D grid of unit weights with 1 % of its edges missing;
* ``rgg``    -- a 3-D random geometric graph of mean degree about 12, with
  vertex weights 1..4 and edge weights 1..16;
* ``rmat``   -- a power-law graph (R-MAT 0.57, 0.19, 0.19, 0.05, edge factor
  16, relabelled at random), unit weights;
* ``banded`` -- an FEM-like pattern of bandwidth 32 with 10 % of entries off
  the band, unit weights.

and of one of the calls:

* ``device``   -- ``partition_device``: CSR in HBM in, part[] in HBM out;
* ``host``     -- ``partition``: host arrays in and out, int64 offsets;
* ``dropin``   -- ``PartitionGraph``: host arrays in and out, int32 offsets;
* ``batch``    -- ``partition_batch``: many graphs of 1k..64k vertices;
* ``serve``    -- ``Server.submit`` / ``wait``: a queue of mixed requests;
* ``evaluate`` -- ``evaluate_device``: cut and heaviest part of a partition.

Every result is a whole number and every path is deterministic, so results
are compared exactly.
"""
import math

import numpy as np
import torch  # before the package: one HIP runtime per process

import hunyuansc25_amd as hgp

#: Degrees and weights of the graph kinds.
RGG_DEGREE = 12.0
BAND = 32
EDGE_FACTOR = 16
RMAT_ABC = (0.57, 0.19, 0.19)


def listed():
    return [
        # The smallest earnest call of the drop-in entry point: a program that
        # partitions a small mesh from its own host arrays; launches and the
        # host's waits are all of it.
        {"name": "dropin_mesh_64x64_k8", "call": "dropin", "graph": "mesh", "rows": 64, "cols": 64, "k": 8},
        # The 256 x 256 mesh of the configurations, resident in HBM: many
        # levels, each of them small.
        {"name": "device_mesh_256x256_k8", "call": "device", "graph": "mesh", "rows": 256, "cols": 256, "k": 8},
        # A large mesh of odd sides, split among many parts.
        {"name": "device_mesh_1023x1537_k96", "call": "device", "graph": "mesh", "rows": 1023, "cols": 1537, "k": 96},
        # The weighted random geometric graph of the configurations.
        {"name": "device_rgg_2p20_k64", "call": "device", "graph": "rgg", "n": 1 << 20, "k": 64},
        # A weighted graph of a simulation's own host arrays, odd sizes: the
        # upload, the checks of the arrays and the download count too.
        {"name": "host_rgg_100003_k12", "call": "host", "graph": "rgg", "n": 100003, "k": 12},
        # An FEM matrix pattern: no hub rows, every row of about 70 entries.
        {"name": "device_banded_200003_k37", "call": "device", "graph": "banded", "n": 200003, "k": 37},
        # A power-law graph split among more than 256 parts (16-bit part ids).
        {"name": "device_rmat_s17_k1000", "call": "device", "graph": "rmat", "scale": 17, "k": 1000},
        # A power-law graph of ordinary size.
        {"name": "device_rmat_s19_k256", "call": "device", "graph": "rmat", "scale": 19, "k": 256},
        # The headline configuration: 2^22 vertices, 2^26 edges.
        {"name": "device_rmat_s22_k256", "call": "device", "graph": "rmat", "scale": 22, "k": 256},
        # Many independent graphs at once, as a solver farm hands them over.
        {"name": "batch_48_graphs", "call": "batch", "count": 48, "lo": 1000, "hi": 65536},
        # A serving queue under load: requests of 10k..260k vertices, 4 slots.
        {"name": "serve_8_requests", "call": "serve", "count": 8, "lo": 10000, "hi": 262144, "slots": 4},
        # Scoring a partition that a program already has.
        {"name": "evaluate_rmat_s20_k256", "call": "evaluate", "graph": "rmat", "scale": 20, "k": 256},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    call = rng.choice(["device", "device", "device", "device", "dropin", "host", "batch", "serve", "evaluate"])
    if call == "batch":
        lo = _log_int(rng, 1000, 4000)
        return {"call": call, "count": rng.randint(8, 48), "lo": lo, "hi": _log_int(rng, 16384, 65536)}
    if call == "serve":
        return {"call": call, "count": rng.randint(3, 8), "lo": _log_int(rng, 10000, 30000),
                "hi": _log_int(rng, 60000, 262144), "slots": rng.randint(2, 6)}
    # vertices of a single graph, over the logarithm of each call's range
    n = {"device": lambda: _log_int(rng, 4000, 1500000), "dropin": lambda: _log_int(rng, 2000, 60000),
         "host": lambda: _log_int(rng, 2000, 200000), "evaluate": lambda: _log_int(rng, 30000, 1000000)}[call]()
    case = {"call": call, "graph": rng.choice(["mesh", "rgg", "rmat", "banded"])}
    if case["graph"] == "mesh":
        case["rows"] = max(2, int(round(math.sqrt(n) * rng.uniform(0.4, 1.0))))
        case["cols"] = max(2, n // case["rows"])
    elif case["graph"] == "rmat":
        case["scale"] = max(11, int(round(math.log2(n))))
    else:
        case["n"] = n if case["graph"] == "rgg" else min(n, 300000)
    # at least about 50 vertices a part, 2..1024 parts
    case["k"] = _log_int(rng, 2, max(3, min(1024, n // 50)))
    return case


# ---------------------------------------------------------------- graphs (device tensors)

def _csr(n, lo, hi):
    """Symmetric CSR with sorted rows of the distinct pairs lo < hi."""
    key, _ = torch.sort(torch.cat([lo * n + hi, hi * n + lo]))
    u = key // n
    xadj = torch.zeros(n + 1, dtype=torch.int64, device=key.device)
    xadj[1:] = torch.cumsum(torch.bincount(u, minlength=n), 0)
    return xadj, (key - u * n).to(torch.int32)


def _unit(xadj, adjncy):
    """The graph with unit weights (the device entry points take arrays)."""
    return xadj, adjncy, torch.ones(xadj.numel() - 1, dtype=torch.int32, device="cuda"), torch.ones_like(adjncy)


def _mesh(rows, cols, gen):
    v = torch.arange(rows * cols, device="cuda").reshape(rows, cols)
    lo = torch.cat([v[:, :-1].reshape(-1), v[:-1].reshape(-1)])
    hi = torch.cat([v[:, 1:].reshape(-1), v[1:].reshape(-1)])
    keep = torch.rand(lo.numel(), device="cuda", generator=gen) >= 0.01
    return _unit(*_csr(rows * cols, lo[keep], hi[keep]))


def _rmat(scale, gen):
    n, edges = 1 << scale, EDGE_FACTOR << scale
    a, b, c = RMAT_ABC
    pairs = torch.empty(0, dtype=torch.int64, device="cuda")
    while pairs.numel() < edges:
        want = int(1.25 * (edges - pairs.numel())) + 1024
        u = torch.zeros(want, dtype=torch.int64, device="cuda")
        v = torch.zeros(want, dtype=torch.int64, device="cuda")
        for _ in range(scale):
            r = torch.rand(want, device="cuda", generator=gen)
            u = 2 * u + (r >= a + b)
            v = 2 * v + (((r >= a) & (r < a + b)) | (r >= a + b + c))
        ok = u != v
        new = torch.minimum(u, v)[ok] * n + torch.maximum(u, v)[ok]
        pairs = torch.unique(torch.cat([pairs, new]))
    if pairs.numel() > edges:   # the same number of edges for every seed
        drop = torch.randperm(pairs.numel(), device="cuda", generator=gen)[: pairs.numel() - edges]
        keep = torch.ones(pairs.numel(), dtype=torch.bool, device="cuda")
        keep[drop] = False
        pairs = pairs[keep]
    name = torch.randperm(n, device="cuda", generator=gen)
    u, v = name[pairs // n], name[pairs % n]
    return _unit(*_csr(n, torch.minimum(u, v), torch.maximum(u, v)))


def _graph(case, seed):
    """(xadj, adjncy, vwgt, adjwgt) as device tensors."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    kind = case["graph"]
    if kind == "mesh":
        return _mesh(case["rows"], case["cols"], gen)
    if kind == "rmat":
        return _rmat(case["scale"], gen)
    n = case["n"]
    if kind == "rgg":
        g = hgp.gen_rgg3d(n, hgp.rgg_radius(n, RGG_DEGREE), seed=seed, vw=(1, 4), ew=(1, 16))
        return tuple(torch.from_numpy(t).cuda() for t in g)
    x, a, _, _ = hgp.gen_banded(n, BAND, 0.1, seed=seed)
    return _unit(torch.from_numpy(x).cuda(), torch.from_numpy(a).cuda())


def _host(g):
    return tuple(t.cpu().numpy() for t in g)


def _sizes(case):
    """Vertex counts of a batch or a queue, spread evenly over the logarithm."""
    s = np.geomspace(case["lo"], case["hi"], case["count"]).astype(np.int64)
    return [int(x) for x in s[::-1]]


# ---------------------------------------------------------------- preparation

class _Session:
    """A server and the requests that a program keeps sending it."""

    def __init__(self, slots, requests):
        self.server = hgp.Server(slots=slots, budget_bytes=64 << 30)
        self.requests = requests

    def __del__(self):
        self.server.close()


def _batch(case, seed):
    graphs, ks = [], []
    for i, n in enumerate(_sizes(case)):
        side = max(2, int(round(math.sqrt(n))))
        graphs.append([lambda: hgp.gen_grid2d(side, max(2, n // side)),
                       lambda: hgp.gen_rgg3d(n, hgp.rgg_radius(n, RGG_DEGREE), seed=seed + i),
                       lambda: hgp.gen_banded(n, BAND, 0.1, seed=seed + i)][i % 3]())
        ks.append([2, 4, 8, 16, 32, 64][(i // 3) % 6])
    return graphs, ks


def _requests(case, seed):
    out = []
    for i, n in enumerate(_sizes(case)):
        kind = {"graph": "rmat", "scale": int(round(math.log2(n)))} if i % 2 == 0 else {"graph": "rgg", "n": n}
        out.append((_host(_graph(kind, seed + i)), 8 << (i % 7)))
    return out


def prepare(case, seed):
    call = case["call"]
    state = {"case": case, "seed": seed}
    if call == "batch":
        state["graphs"], state["ks"] = _batch(case, seed)
    elif call == "serve":
        state["session"] = _Session(case["slots"], _requests(case, seed))
    else:
        g = _graph(case, seed)
        n = g[0].numel() - 1
        if call == "host":
            state["graph"] = _host(g)
        elif call == "dropin":
            x, a, vw, aw = _host(g)
            state["graph"] = (x.astype(np.int32), a, vw, aw)
        else:
            state["graph"] = g
            state["n"] = n
            state["ptr"] = [t.data_ptr() for t in g]
            state["part"] = torch.zeros(n, dtype=torch.int32, device="cuda")
            if call == "evaluate":
                # runs of vertices with a fifth of them misplaced
                gen = torch.Generator(device="cuda")
                gen.manual_seed(seed + 1)
                k = case["k"]
                block = torch.arange(n, device="cuda") * k // n
                other = torch.randint(0, k, (n,), device="cuda", generator=gen)
                mixed = torch.rand(n, device="cuda", generator=gen) < 0.2
                state["part"].copy_(torch.where(mixed, other, block))
                state["out"] = torch.zeros(4, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()   # the library works on a stream of its own
    return state


# ---------------------------------------------------------------- one pass

def run(state):
    case, seed = state["case"], state["seed"]
    call = case["call"]
    if call == "device":
        x, a, vw, aw = state["ptr"]
        st = hgp.partition_device(state["n"], x, a, vw, aw, case["k"], state["part"].data_ptr(), seed=seed)
        return {"part": state["part"], "cut": st["cut"], "max_pwgt": st["max_pwgt"]}
    if call == "host":
        x, a, vw, aw = state["graph"]
        part, st = hgp.partition(x, a, case["k"], vw, aw, seed=seed)
        return {"part": part, "cut": st["cut"], "max_pwgt": st["max_pwgt"]}
    if call == "dropin":
        x, a, vw, aw = state["graph"]
        return hgp.PartitionGraph(len(x) - 1, x, a, vw, aw, case["k"], None, 1.03)
    if call == "batch":
        parts, stats = hgp.partition_batch(state["graphs"], state["ks"], seed=seed)
        return {"parts": parts, "cuts": np.array([st["cut"] for st in stats])}
    if call == "serve":
        s = state["session"]
        tickets = [s.server.submit(x, a, k, vw, aw, seed=seed) for (x, a, vw, aw), k in s.requests]
        done = [s.server.wait(t) for t in tickets]
        return {"parts": [d[0] for d in done], "cuts": np.array([d[1]["cut"] for d in done])}
    x, a, vw, aw = state["ptr"]
    hgp.evaluate_device(state["n"], x, a, aw, vw, state["part"].data_ptr(), case["k"], state["out"].data_ptr())
    return state["out"]


# ---------------------------------------------------------------- cost, tolerance, reference

def _entries(graph, n):
    """Directed entries of a graph of n vertices."""
    return {"mesh": 3.96, "rgg": RGG_DEGREE, "rmat": 2.0 * EDGE_FACTOR, "banded": 2.2 * BAND}[graph] * n


def _bytes(graph, n):
    """The graph read once (offsets, neighbours, weights) and part[] written."""
    return 8.0 * (n + 1) + 8.0 * _entries(graph, n) + 4.0 * n + 4.0 * n


def work(case):
    if case["call"] == "batch":
        jobs = [(["mesh", "rgg", "banded"][i % 3], n) for i, n in enumerate(_sizes(case))]
    elif case["call"] == "serve":
        jobs = [("rmat", 1 << int(round(math.log2(n)))) if i % 2 == 0 else ("rgg", n)
                for i, n in enumerate(_sizes(case))]
    else:
        n = case.get("n") or (1 << case["scale"] if "scale" in case else case["rows"] * case["cols"])
        jobs = [(case["graph"], n)]
    # one operation an entry: the weight that it adds to a part's connectivity
    return {"bytes": sum(_bytes(g, n) for g, n in jobs), "flops": sum(_entries(g, n) for g, n in jobs)}


def tolerance(case):
    return "exact"


def exact(case, seed):
    """The evaluation counted with plain torch; a partition has no reference
    value of its own."""
    if case["call"] != "evaluate":
        return None
    state = prepare(case, seed)
    x, a, vw, aw = state["graph"]
    part, n = state["part"].long(), state["n"]
    row = torch.repeat_interleave(torch.arange(n, device="cuda"), x[1:] - x[:-1])
    cut = int((aw.long() * (part[row] != part[a.long()])).sum()) // 2
    pw = torch.zeros(case["k"], dtype=torch.int64, device="cuda")
    pw.index_add_(0, part, vw.long())
    return torch.tensor([cut, int(pw.max()), 0, 0], dtype=torch.int64)
