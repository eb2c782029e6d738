"""The work a user of this library has it do, as cases that can be timed and checked.

Every case is a graph and one call on it through the public Python entry
points: a query of an engine (`Engine.run`) or a batch of queries
(`batch.run_batch`).  Three families of graphs, each with the sizes that the
benchmark, the tests and the batched workload use:

  rmat   `Graph.rmat`: social-network-like, 2^scale vertices, few wide frontiers
  grid   `Graph.grid`: road-like n x n lattice with 10 % of the edges missing,
         thousands of narrow frontiers
  edges  `Graph.from_edges`: a caller's own skewed edge list, with a vertex
         count that is no power of two

Ranges that the listed cases stand for and that `draw` covers:

  BFS    rmat scales 12-24, edge factors 8-24; lattices of 256^2 to 1500^2
  SSSP   rmat scales 12-24, edge factors 8-16, weights up to 100, 1000 or
         100 000 (they fit 8, 16 or 32 bits); edge lists; lattices with
         weights up to 1000 and the bucket width that suits them
  CC     directed label propagation, rmat scales 12-23 and edge lists
  WCC    symmetrized rmat, scales 12-24
  PR     20 iterations, rmat scales 12-24 and edge lists; the social-follower
         shape (scale 25, edge factor 44) is the largest
  batch  BFS and SSSP queries from uniform roots over rmat and lattice graphs
         of uneven size

Engines take the GPU schedule and the tuning table's options where the table
has an entry for the graph's size class, as the benchmark does.  Small results
come back to host memory, where such a caller reads them; large ones stay in
HBM and are read through `cg_engine_result_device`.
"""
import ctypes
import random

import numpy as np
import torch

import cggraph_amd as cg
from cggraph_amd import autotune, batch

BFS, SSSP, CC, PR = 0, 1, 2, 3
ALGORITHM = {"bfs": BFS, "sssp": SSSP, "cc": CC, "wcc": CC, "pr": PR}
PR_ITERATIONS, PR_DAMPING = 20, 0.85
HOST_RESULT_V = 1 << 20  # results of up to this many vertices go to host memory


def listed():
    return [
        # one query on a small graph: launches and waits are all there is
        {"name": "bfs_rmat12", "do": "bfs", "graph": "rmat", "scale": 12, "edge_factor": 8, "to_host": True},
        # the reference's CPU-runnable configuration
        {"name": "bfs_rmat18", "do": "bfs", "graph": "rmat", "scale": 18, "edge_factor": 16, "to_host": False},
        # BFS on a graph far beyond the caches
        {"name": "bfs_rmat24", "do": "bfs", "graph": "rmat", "scale": 24, "edge_factor": 16, "to_host": False},
        # hop counts over a road-like network: about 1500 narrow levels
        {"name": "bfs_grid1000", "do": "bfs", "graph": "grid", "n": 1000, "max_weight": 0, "to_host": True},
        # SSSP on a caller's own edge list, default options, result read on the host
        {"name": "sssp_edges1m", "do": "sssp", "graph": "edges", "V": 1000003, "edge_factor": 12, "max_weight": 1000,
         "to_host": True},
        # the headline benchmark
        {"name": "sssp_rmat24", "do": "sssp", "graph": "rmat", "scale": 24, "edge_factor": 16, "max_weight": 100,
         "to_host": False},
        # routing distances over a road-like network, bucketed
        {"name": "sssp_grid1500", "do": "sssp", "graph": "grid", "n": 1500, "max_weight": 1000, "sssp_delta": 3000,
         "to_host": False},
        # label propagation over a directed graph (the reference's CC)
        {"name": "cc_rmat22", "do": "cc", "graph": "rmat", "scale": 22, "edge_factor": 16, "to_host": False},
        # components of an undirected graph
        {"name": "wcc_rmat24", "do": "wcc", "graph": "rmat", "scale": 24, "edge_factor": 16, "to_host": False},
        # PageRank of an ordinary graph, ranks read on the host
        {"name": "pr_edges300k", "do": "pr", "graph": "edges", "V": 300007, "edge_factor": 16, "to_host": True},
        # PageRank of a large social follower graph
        {"name": "pr_rmat25", "do": "pr", "graph": "rmat", "scale": 25, "edge_factor": 44, "to_host": False},
        # many queries over graphs of uneven size in one call (the batched
        # benchmark's 13 graphs, four queries on each)
        {"name": "batch_mixed", "do": "batch", "queries": 52, "scale_lo": 14, "scale_hi": 22, "side_lo": 256,
         "sides": 4},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    do = rng.choice(["bfs", "bfs", "sssp", "sssp", "cc", "wcc", "pr", "batch"])
    if do == "batch":
        lo = rng.randint(12, 17)
        return {"do": "batch", "queries": rng.randint(8, 48), "scale_lo": lo, "scale_hi": lo + rng.randint(1, 4),
                "side_lo": rng.randint(100, 300), "sides": rng.randint(1, 3)}
    c = {"do": do}
    kind = rng.choice({"bfs": ["rmat", "rmat", "grid"], "sssp": ["rmat", "edges", "grid"], "cc": ["rmat", "edges"],
                       "wcc": ["rmat"], "pr": ["rmat", "edges"]}[do])
    c["graph"] = kind
    if kind == "rmat":
        top = {"bfs": 24, "sssp": 24, "cc": 23, "wcc": 24, "pr": 24}[do]
        c["scale"] = rng.randint(12, top)
        c["edge_factor"] = rng.randint(8, 16 if do != "bfs" or c["scale"] == 24 else 24)
        V = 1 << c["scale"]
    elif kind == "edges":
        V = c["V"] = _log_uniform(rng, 5000, 1500000) | 1
        c["edge_factor"] = rng.randint(6, 16)
    else:
        c["n"] = _log_uniform(rng, 256, 1500)
        V = c["n"] ** 2
    if do == "sssp":
        c["max_weight"] = rng.choice([100, 1000, 100000]) if kind != "grid" else 1000
        if kind == "grid":
            c["sssp_delta"] = 3000
    elif kind == "grid":
        c["max_weight"] = 0
    c["to_host"] = V <= HOST_RESULT_V and rng.random() < 0.5
    return c


def _edge_list(case, seed):
    """A skewed edge list on the GPU: R-MAT quadrants over the next power of
    two, scaled down to V vertices.  (src, dst) as int64."""
    V = case["V"]
    levels = (V - 1).bit_length()
    m = V * case["edge_factor"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    src = torch.zeros(m, dtype=torch.int64, device="cuda")
    dst = torch.zeros_like(src)
    for _ in range(levels):
        x = torch.rand(m, device="cuda", generator=gen)
        src = src * 2 + (x >= 0.76)
        dst = dst * 2 + (((x >= 0.57) & (x < 0.76)) | (x >= 0.95))
    return (src * V) >> levels, (dst * V) >> levels, gen


def _graph(case, seed):
    do = case["do"]
    max_weight = case.get("max_weight", 0)
    weights = (1, max_weight) if max_weight else None
    if case["graph"] == "rmat":
        return cg.Graph.rmat(case["scale"], case["edge_factor"], seed=seed, weights=weights, symmetrize=do == "wcc")
    if case["graph"] == "grid":
        return cg.Graph.grid(case["n"], 0.1, seed=seed, weights=weights)
    src, dst, gen = _edge_list(case, seed)
    w = None
    if max_weight:
        w = torch.randint(1, max_weight + 1, src.shape, device="cuda", generator=gen, dtype=torch.int32)
        w = w.cpu().numpy().view(np.uint32)
    as_u32 = lambda t: t.to(torch.int32).cpu().numpy().view(np.uint32)  # noqa: E731
    return cg.Graph.from_edges(case["V"], as_u32(src), as_u32(dst), w)


class _DeviceResult:
    """An engine's result in HBM, as an array other libraries can view."""

    def __init__(self, engine, dtype):
        self._engine = engine  # the memory is the engine's
        p = ctypes.c_void_p()
        if cg.lib().cg_engine_result_device(engine._h, ctypes.byref(p)) != 0:
            raise RuntimeError("cg_engine_result_device failed")
        self.__cuda_array_interface__ = {"shape": (engine.V,), "typestr": dtype, "data": (p.value, False),
                                         "version": 3}


def prepare(case, seed):
    if case["do"] == "batch":
        sides = [case["side_lo"] << i for i in range(case["sides"])]
        n = case["queries"]
        graphs, on, algorithms, roots = batch.mixed_workload(
            n - n // 2, n // 2, range(case["scale_lo"], case["scale_hi"] + 1), sides, seed=seed)
        return {"batch": (on, algorithms, roots), "graphs": graphs, "options": autotune.best_options("batch/mixed")}
    algorithm = ALGORITHM[case["do"]]
    g = _graph(case, seed)
    info = g.info()
    root, options = info["max_outdeg_vertex"], {}
    if case["graph"] == "grid":
        root = random.Random(seed).randrange(info["V"])
        options["sssp_delta"] = case.get("sssp_delta", 0)
    elif algorithm in (BFS, SSSP):
        options = autotune.best_options(autotune.engine_signature("rmat", algorithm, info["V"], info["E"]))
    engine = cg.Engine(g, algorithm, **options)
    return {"engine": engine, "root": root, "to_host": case["to_host"], "dtype": "<f4" if algorithm == PR else "<i4"}


def run(state):
    if "batch" in state:
        on, algorithms, roots = state["batch"]
        values, _ = batch.run_batch(on, algorithms, roots, **state["options"])
        return [v.view(np.int32) for v in values]
    engine = state["engine"]
    if state["to_host"]:
        values, _ = engine.run(state["root"])
        return values if state["dtype"] == "<f4" else values.view(np.int32)
    engine.run(state["root"], copy_out=False)
    return torch.as_tensor(_DeviceResult(engine, state["dtype"]), device="cuda")


def _size(case):
    """(vertices, edges) before parallel edges are merged."""
    if case["graph"] == "rmat":
        V = 1 << case["scale"]
        return V, V * case["edge_factor"] * (2 if case["do"] == "wcc" else 1)
    if case["graph"] == "grid":
        return case["n"] ** 2, int(3.6 * case["n"] ** 2)
    return case["V"], case["V"] * case["edge_factor"]


def work(case):
    """Each edge and each row once (for PageRank once in every iteration: the
    ranks of the one before decide), and the values once; an operation per
    edge.  A BFS that goes bottom-up and the sampled components need not look
    at every edge, so their rate can pass a streaming one."""
    if case["do"] == "batch":
        one = [work({"do": "sssp", "graph": "rmat", "scale": s, "edge_factor": 16})
               for s in range(case["scale_lo"], case["scale_hi"] + 1)]
        one += [work({"do": "sssp", "graph": "grid", "n": case["side_lo"] << i}) for i in range(case["sides"])]
        share = case["queries"] / len(one)
        return {k: share * sum(w[k] for w in one) for k in ("bytes", "flops")}
    V, E = _size(case)
    if case["do"] == "pr":
        return {"bytes": PR_ITERATIONS * (4.0 * E + 8.0 * (V + 1) + 8.0 * V), "flops": PR_ITERATIONS * (E + 3.0 * V)}
    return {"bytes": (8.0 if case["do"] == "sssp" else 4.0) * E + 8.0 * (V + 1) + 4.0 * V, "flops": 1.0 * E}


# ---- PageRank in 64 bits, without the library ----

_GOLDEN = 0x9E3779B97F4A7C15


def _signed(x):
    x &= (1 << 64) - 1
    return x - (1 << 64) if x >> 63 else x


def _mix64(z):
    """SplitMix64's finaliser on int64 tensors (products wrap; the shifts are logical)."""
    z = (z ^ ((z >> 30) & ((1 << 34) - 1))) * _signed(0xBF58476D1CE4E5B9)
    z = (z ^ ((z >> 27) & ((1 << 37) - 1))) * _signed(0x94D049BB133111EB)
    return z ^ ((z >> 31) & ((1 << 33) - 1))


def _rmat_list(scale, edge_factor, seed, block=1 << 26):
    """The edges `Graph.rmat` generates, from its specification: level l of
    edge i takes a 32-bit half of draw(i, l // 2) and a quadrant by integer
    thresholds.  (src, dst) as int32."""
    m = edge_factor << scale
    key = int(_mix64(torch.tensor(_signed(seed * _GOLDEN + 0x5851F42D4C957F2D))))
    t_a, t_ab, t_abc = (int(p * 4294967296.0) for p in (0.57, 0.57 + 0.19, 0.57 + 0.19 + 0.19))
    src = torch.empty(m, dtype=torch.int32, device="cuda")
    dst = torch.empty_like(src)
    for lo in range(0, m, block):
        i = torch.arange(lo, min(m, lo + block), dtype=torch.int64, device="cuda") * 16
        s, d = torch.zeros_like(i), torch.zeros_like(i)
        for level in range(scale):
            if level % 2 == 0:
                r = _mix64((i + (level // 2 + 1)) * _signed(_GOLDEN) + key)
            x = (r >> (32 * (level & 1))) & 0xFFFFFFFF
            s = s * 2 + (x >= t_ab)
            d = d * 2 + (((x >= t_a) & (x < t_ab)) | (x >= t_abc))
        src[lo:lo + block] = s
        dst[lo:lo + block] = d
    return src, dst


def exact(case, seed):
    """PageRank's ranks from 64-bit arithmetic: a row's contributions are added
    as 60-bit fixed point, whose sums do not depend on their order.  The other
    algorithms' results are whole numbers."""
    if case["do"] != "pr":
        return None
    if case["graph"] == "rmat":
        V = 1 << case["scale"]
        src, dst = _rmat_list(case["scale"], case["edge_factor"], seed)
    else:
        V = case["V"]
        src, dst, _ = _edge_list(case, seed)
    bits = (V - 1).bit_length()
    edge = (dst.to(torch.int64) << bits) | src  # by destination, then source
    del src, dst
    mask = (1 << bits) - 1
    edge = edge[(edge >> bits) != (edge & mask)]  # no self-loops
    edge = edge.sort().values
    first = torch.ones(edge.numel(), dtype=torch.bool, device="cuda")
    first[1:] = edge[1:] != edge[:-1]  # parallel edges merged
    edge = edge[first]
    del first
    row_end = torch.searchsorted(edge, torch.arange(1, V + 1, device="cuda") << bits)
    src = edge & mask
    del edge
    degree = torch.bincount(src, minlength=V).clamp(min=1).double()
    rank = torch.full((V,), 1.0 / V, dtype=torch.float64, device="cuda")
    for _ in range(PR_ITERATIONS):
        total = (rank / degree * 2.0 ** 60).to(torch.int64)[src].cumsum(0)
        at = torch.cat([total.new_zeros(1), total])[row_end]
        total = torch.diff(at, prepend=at.new_zeros(1))
        rank = (1 - PR_DAMPING) / V + PR_DAMPING * (total.double() * 2.0 ** -60)
    return rank.cpu().numpy() if case["to_host"] else rank
