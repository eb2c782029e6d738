"""The batch's level loop, on a graph that neither clusters nor engines take
(more than 2^18 edges, rows above 64, no hub): its launch shapes, buckets, hub
deferral and the two-kernel form past 4096 queries, bit-exact against the
oracle."""
import numpy as np
import pytest

import cggraph_amd as cg
from cggraph_amd import batch

pytestmark = pytest.mark.gpu
BFS, SSSP = 0, 1


@pytest.fixture(scope="module")
def graph(oracle):
    rng = np.random.default_rng(1)
    V, m = 2000, 300_000
    og = oracle.csr_build(V, rng.integers(0, V, m).astype(np.uint32), rng.integers(0, V, m).astype(np.uint32))
    og.weight = rng.integers(1, 1001, og.E).astype(np.uint32)
    deg = np.diff(og.offsets.astype(np.int64)).max()
    assert og.E > 1 << 18 and 64 < deg < 16 * og.E // V
    h = cg.Graph.from_csr(og.offsets, og.dest, og.weight)
    yield og, h
    h.close()


def check(oracle, og, h, algs, roots, **opt):
    outs, st = batch.run_batch([h] * len(roots), algs, roots, **opt)
    refs = {}
    for a, r, got in zip(algs, roots, outs):
        if (a, r) not in refs:
            refs[a, r] = oracle.bfs(og, r) if a == BFS else oracle.sssp(og, r)
        assert np.array_equal(got, refs[a, r]), (a, r, opt)
    assert st["edges_traversed"] == sum(oracle.reached_edges(og, refs[q]) for q in zip(algs, roots))
    assert st["heavy_iterations"] == 0


@pytest.mark.parametrize("block,grid,levels,delta,group,hub", [
    (64, 1, 1, 0, 64, 0), (1024, 512, 32, 0, 1, 0), (256, 64, 8, 1, 16, 0), (256, 2048, 16, 50, 32, 0),
    (512, 128, 4, 10**7, 7, 0), (256, 256, 8, 0, 32, 150), (256, 256, 8, 30, 32, 150), (256, 256, 8, 0, 32, 1)])
def test_shapes(oracle, graph, block, grid, levels, delta, group, hub):
    og, h = graph
    check(oracle, og, h, [BFS, SSSP] * 4, [0, 0, 17, 17, 1999, 1999, 450, 3], batch_block=block, batch_grid=grid,
          batch_levels=levels, sssp_delta=delta, batch_group=group, hub_degree=hub, hub_delta=20)


@pytest.mark.parametrize("delta", [0, 100])
@pytest.mark.parametrize("n", [4096, 4097])
def test_many_queries(oracle, graph, n, delta):
    og, h = graph
    check(oracle, og, h, [i % 2 for i in range(n)], [i % 37 for i in range(n)], batch_levels=8, batch_grid=256,
          sssp_delta=delta)
