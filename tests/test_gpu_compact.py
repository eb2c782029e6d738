"""Frontier compaction in slices of 4 and of 16 vertices (csrc/traverse.hip):
either side of the sizes where the finer ones and the smaller workgroups end;
the first frontier and the default tiers sized by the graph.  Depths,
distances and labels bit-exact against the oracle."""
import numpy as np
import pytest

import cggraph_amd as cg

pytestmark = pytest.mark.gpu

BFS, SSSP, CC = 0, 1, 2


def skewed(oracle, V, E, weights, seed):
    rng = np.random.default_rng(seed)
    src = (V * rng.random(E) ** 4).astype(np.uint32)  # a few vertices send most edges
    dst = rng.integers(0, V, E).astype(np.uint32)
    src[: V // 8] = 0  # one vertex above every tier
    og = oracle.csr_build(V, src, dst)
    og.weight = rng.integers(1, weights + 1, og.E).astype(np.uint32)
    return og


@pytest.mark.parametrize("V", [65, 4097, 2**18 - 63, 2**18, 2**18 + 1, 2**20, 2**20 + 1, 2**22, 2**22 + 1])
@pytest.mark.parametrize("hub", [0, 128])
def test_slices(oracle, V, hub):
    og = skewed(oracle, V, (3 if V < 2**20 else 1) * V + 70000, 100, V % 97)
    g = cg.Graph.from_csr(og.offsets, og.dest, og.weight)
    e = cg.Engine(g, SSSP, hub_degree=hub, hub_delta=3)
    for root in (0, 1):
        got, _ = e.run(root)
        assert np.array_equal(got, oracle.sssp(og, root)), (V, root)
    e.close()
    if not hub:
        e = cg.Engine(g, BFS)
        assert np.array_equal(e.run(1)[0], oracle.bfs(og, 1)), V
        e.close()
        e = cg.Engine(g, CC)
        assert np.array_equal(e.run(0)[0], oracle.cc_directed(og)), V
        e.close()
    g.close()


def test_tiers(oracle):
    """Chunks by the graph's size, by the caller and at the first frontier."""
    og = skewed(oracle, 30011, 900000, 1000, 5)
    g = cg.Graph.from_csr(og.offsets, og.dest, og.weight)
    for opts in ({}, {"bin_wave": 600}, {"bin_chunk": 64, "bin_wave": 64, "chunk_edges": 1}, {"chunk_edges": 100000},
                 {"sssp_delta": 200}):
        e = cg.Engine(g, SSSP, **opts)
        for root in (0, 17):
            assert np.array_equal(e.run(root)[0], oracle.sssp(og, root)), (opts, root)
        e.close()
