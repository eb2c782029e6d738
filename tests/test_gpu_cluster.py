"""Level cluster (csrc/cluster.hip): the GPU schedule runs narrow frontiers
inside one launch and hands wide ones back.  Bit-exact against the CPU oracle
where that can go wrong: rows around an entry's 256 edges, frontiers that
outgrow a level and shrink again, bucketed runs, several roots on an engine."""
import numpy as np
import pytest

import cggraph_amd as cg

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


@pytest.mark.parametrize("delta", [1, 30])
def test_full_far_list(oracle, delta):
    """A bucketed run whose far lists outgrow their room hands back a frontier
    of waiting vertices only: a hub reaches 200 000 leaves (16 lists hold
    131 072), each with a chain of its own, all beyond the first bucket."""
    leaves, rng = 200_000, np.random.default_rng(delta)
    mid = 5000  # the root's row stays short, so the run starts in the cluster
    src = [np.zeros(50, np.int64), np.repeat(np.arange(1, 51), 60), np.repeat(np.arange(51, 3051), 66)]
    dst = [np.arange(1, 51), np.arange(51, 3051), mid + np.arange(198_000)]
    src.append(mid + np.arange(leaves))
    dst.append(mid + leaves + np.arange(leaves))
    V = mid + 2 * leaves
    og = weighted(oracle, V, np.concatenate(src), np.concatenate(dst), 7)
    og.weight = rng.integers(40, 60_000, og.E).astype(np.uint32)
    check(oracle, og, SSSP, [0, 60, mid], sssp_delta=delta * 1000)
