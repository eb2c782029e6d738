"""Level cluster (csrc/cluster.hip): the GPU schedule runs narrow frontiers
inside one launch and hands wide ones back.  Bit-exact against the CPU oracle
where that can go wrong: rows around an entry's 256 edges, frontiers that
outgrow a level and shrink again, bucketed runs, several roots on an engine."""
import numpy as np
import pytest

import cggraph_amd as cg
from cggraph_amd import batch

pytestmark = pytest.mark.gpu
BFS, SSSP, CC = 0, 1, 2


def weighted(oracle, V, src, dst, seed, wmax=100):
    g = oracle.csr_build(V, np.asarray(src, np.uint32), np.asarray(dst, np.uint32))
    g.weight = np.random.default_rng(seed).integers(1, wmax + 1, g.E).astype(np.uint32)
    return g


def check(oracle, og, alg, roots, **opt):
    g = cg.Graph.from_csr(og.offsets, og.dest, og.weight)
    e = cg.Engine(g, alg, **opt)
    for i, r in enumerate(list(roots) + list(roots)[:1]):
        ref = oracle.bfs(og, r) if alg == BFS else (oracle.sssp(og, r) if alg == SSSP else oracle.cc_directed(og))
        got, st = e.run(r, copy_out=(i % 2 == 0))
        got = e.result() if got is None else got
        assert np.array_equal(got, ref), (alg, r, opt)
        if alg != CC:
            assert st["edges_traversed"] == oracle.reached_edges(og, ref), (alg, r, opt)
    e.close()
    g.close()


@pytest.mark.parametrize("n", [1, 2, 9, 63, 300])
def test_lattices(oracle, n):
    og = oracle.grid_graph(n, 0.1, seed=n)
    roots = sorted({0, n * n // 2, n * n - 1})
    check(oracle, og, BFS, roots)
    for delta in (0, 1 if n < 64 else 100, 3000, 4_000_000_000):
        check(oracle, og, SSSP, roots, sssp_delta=delta)


@pytest.mark.parametrize("deg", [255, 256, 257, 512, 513, 30000])
def test_row_lengths(oracle, deg):
    """A hub whose row is cut into entries, a chain behind its last leaf."""
    V = deg + 402
    src = [0] * deg + list(range(deg, deg + 400))
    dst = list(range(1, deg + 1)) + list(range(deg + 1, deg + 401))
    og = weighted(oracle, V, src, dst, deg)
    for alg in (BFS, SSSP, CC):
        check(oracle, og, alg, [0, deg, V - 1])


@pytest.mark.parametrize("wmax", [1, 200, 60000, 10**6])
def test_frontier_handed_back_and_taken_again(oracle, wmax):
    """A 20-ary tree whose fourth level has 160 000 edges (more than one level
    of the cluster holds), whose leaves all meet in one vertex, and a chain
    behind it: narrow, wide and narrow again; with weights below 2^8, 2^16
    and 2^32, plain and bucketed."""
    f, first = 20, [0, 1, 21, 421, 8421, 168421]
    src, dst = [], []
    for level in range(4):
        for i in range(first[level + 1] - first[level]):
            src += [first[level] + i] * f
            dst += range(first[level + 1] + i * f, first[level + 1] + (i + 1) * f)
    leaves, end = range(first[4], first[5]), first[5]
    src += list(leaves) + list(range(end, end + 600))
    dst += [end] * len(leaves) + list(range(end + 1, end + 601))
    og = weighted(oracle, end + 601, src, dst, wmax, wmax)
    roots = [0, 1, end]
    check(oracle, og, BFS, roots)
    check(oracle, og, SSSP, roots)
    check(oracle, og, SSSP, roots, sssp_delta=max(1, wmax // 3))
    check(oracle, og, SSSP, roots, hub_degree=20, hub_delta=1)


@pytest.mark.parametrize("m", [65000, 65536, 66000])
def test_whole_query_in_one_level_budget(oracle, m):
    """Graphs around the edge count up to which every frontier is the cluster's."""
    rng = np.random.default_rng(m)
    V = 9001
    keys = rng.choice(V * V, m, replace=False)
    og = weighted(oracle, V, keys // V, keys % V, m)
    for alg in (BFS, SSSP, CC):
        check(oracle, og, alg, [0, V - 1])


@pytest.mark.parametrize("scale", [12, 15])
def test_tails(oracle, scale):
    """Skewed graphs: wide frontiers first, the shrinking tail in the cluster."""
    og = oracle.rmat_graph(scale, 16, seed=scale, weights=(1, 1000))
    roots = [oracle.max_outdeg_vertex(og), 1, og.V - 2]
    for alg in (BFS, SSSP, CC):
        check(oracle, og, alg, roots)
    check(oracle, og, SSSP, roots, hub_degree=16, hub_delta=10)
    check(oracle, og, SSSP, roots, sssp_delta=200)


def far_graph(oracle, delta):
    """A root that reaches 198 000 leaves within three steps, each with a vertex
    of its own behind it, at weights far beyond a bucket of width delta."""
    leaves, rng = 200_000, np.random.default_rng(delta)
    mid = 5000  # the root's row stays short, so the run starts in the cluster
    src = [np.zeros(50, np.int64), np.repeat(np.arange(1, 51), 60), np.repeat(np.arange(51, 3051), 66)]
    dst = [np.arange(1, 51), np.arange(51, 3051), mid + np.arange(198_000)]
    src.append(mid + np.arange(leaves))
    dst.append(mid + leaves + np.arange(leaves))
    V = mid + 2 * leaves
    og = weighted(oracle, V, np.concatenate(src), np.concatenate(dst), 7)
    og.weight = rng.integers(40, 60_000, og.E).astype(np.uint32)
    return og, [0, 60, mid]


@pytest.mark.parametrize("delta", [1000, 30000])
def test_full_far_list(oracle, delta):
    """A bucketed run whose far lists outgrow their room (16 lists hold 131 072
    entries) hands back a frontier of waiting vertices only."""
    og, roots = far_graph(oracle, delta)
    check(oracle, og, SSSP, roots, sssp_delta=delta)


@pytest.mark.parametrize("fill", [0, 40])
def test_batch_on_clusters(oracle, fill):
    """Batched queries run from root to end on a cluster: lattices, skewed
    graphs whose frontiers outgrow the queues (with more than 32 queries a
    cluster has 4 workgroups and room for 32 768 entries) and full far lists
    (expanded from the bitmap then), beside queries on engines and in the
    level loop."""
    far, far_roots = far_graph(oracle, 1000)
    ogs = [oracle.rmat_graph(16, 16, seed=5, weights=(1, 1000)), oracle.grid_graph(120, 0.1, seed=3), far,
           oracle.rmat_graph(18, 12, seed=6, weights=(1, 1000))]
    gs = [cg.Graph.from_csr(o.offsets, o.dest, o.weight) for o in ogs]
    roots = [[oracle.max_outdeg_vertex(ogs[0]), 7], [0, 7000], far_roots[:2], [oracle.max_outdeg_vertex(ogs[3]), 3]]
    qs = [(k, a, r) for k in range(4) for a in (BFS, SSSP) for r in roots[k]] + [(1, BFS, 100 + i) for i in range(fill)]
    for opt in ({"sssp_delta": 0}, {"sssp_delta": 1000}, {"sssp_delta": 3000, "batch_engine_v": 0xFFFFFFFF}):
        outs, st = batch.run_batch([gs[k] for k, _, _ in qs], [a for _, a, _ in qs], [r for _, _, r in qs], **opt)
        total = 0
        for (k, a, r), got in zip(qs, outs):
            ref = oracle.bfs(ogs[k], r) if a == BFS else oracle.sssp(ogs[k], r)
            assert np.array_equal(got, ref), (k, a, r, opt)
            total += oracle.reached_edges(ogs[k], ref)
        assert st["edges_traversed"] == total
        on_engines = sum(1 for k, _, _ in qs if ogs[k].V >= 1 << 18 and np.diff(ogs[k].offsets.astype(np.int64)).max() >=
                         16 * max(-(-ogs[k].E // ogs[k].V), 1))
        assert on_engines == 8 and st["heavy_iterations"] == (0 if "batch_engine_v" in opt else on_engines)
    for g in gs:
        g.close()
