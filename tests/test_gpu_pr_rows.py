"""PageRank over blocks of consecutive rows (csrc/pagerank.hip): rows around
the lane / wavefront / chunk limits, blocks of empty rows, ranks written in the
caller's ids by the last sweep.  FP64 oracle; the bound is FP32's rounding
(2^-24 of the total mass per addition along the longest chain, 31 + 6 adds in a
block, 16 + 8 per chunk, over 20 damped iterations: 1e-6 of the mass of 1 with
slack), and run-to-run bit-identity."""
import numpy as np
import pytest

import cggraph_amd as cg

pytestmark = pytest.mark.gpu

PR = 3


def graphs(oracle):
    rng = np.random.default_rng(3)
    deg = [31, 32, 33, 63, 64, 65, 2047, 2048, 2049, 4095, 4096, 4097, 8192, 20481, 1, 0, 2047, 2047, 31, 31]
    V = 4000  # the rows above, then empty ones (more than a block of them), then a few with one edge
    dst = np.concatenate([np.repeat(np.arange(len(deg)), deg), np.arange(V - 100, V)])
    src = rng.integers(0, V, len(dst))
    yield "limits", oracle.csr_build(V, src.astype(np.uint32), dst.astype(np.uint32))
    # the last row of a block takes it to just below twice the block's edges
    deg = np.full(70, 30)
    deg[67:] = 2047
    dst = np.repeat(np.arange(70), deg)
    yield "full block", oracle.csr_build(70, rng.integers(0, 70, len(dst)).astype(np.uint32), dst.astype(np.uint32))
    yield "one edge", oracle.csr_build(2, np.array([1], np.uint32), np.array([0], np.uint32))
    yield "no edge", oracle.csr_build(513, np.zeros(0, np.uint32), np.zeros(0, np.uint32))
    yield "renumbered", oracle.rmat_graph(17, 9, seed=6, weights=None)


@pytest.mark.parametrize("layout,kernel", [(1, 0), (2, 0), (1, 1), (2, 1)])
def test_row_blocks(oracle, layout, kernel):
    for name, og in graphs(oracle):
        g = cg.Graph.from_csr(og.offsets, og.dest)
        for iters in (0, 1, 2, 20):
            e = cg.Engine(g, PR, pr_layout=layout, pr_kernel=kernel, pr_iterations=iters)
            r1, _ = e.run()
            r2, _ = e.run()
            e.close()
            assert np.array_equal(r1.view(np.uint32), r2.view(np.uint32)), (name, iters)
            ref = oracle.pagerank64(og, iters, 0.85)
            l1 = float(np.abs(r1.astype(np.float64) - ref).sum())
            assert l1 <= 1e-6, (name, iters, l1)
        g.close()


def test_pair_groups(oracle):
    """Pair blocking's gather (layout 5): whole groups of 512 edges and the
    ends of tiles, contributions either side of 2^-4 (the wide conversion),
    hot bins in several tiles, ranks in the caller's ids."""
    rng = np.random.default_rng(9)
    cases = []
    for n in (511, 512, 513, 1100):  # everything into vertex 0, which gives half the mass to vertex 1
        cases.append((n, np.arange(n), np.r_[1, np.zeros(n - 1, np.int64)]))
    V = 40001  # three bins, the first in several tiles
    src = (V * rng.random(900001) ** 3).astype(np.int64)
    dst = np.where(rng.random(900001) < 0.9, rng.integers(0, 8192, 900001), rng.integers(0, V, 900001))
    cases.append((V, src, dst))
    for V, src, dst in cases:
        og = oracle.csr_build(V, src.astype(np.uint32), dst.astype(np.uint32))
        g = cg.Graph.from_csr(og.offsets, og.dest)
        for iters in (0, 1, 2, 20):
            e = cg.Engine(g, PR, pr_layout=5, pr_iterations=iters)
            r1, _ = e.run()
            r2, _ = e.run()
            e.close()
            assert np.array_equal(r1.view(np.uint32), r2.view(np.uint32)), (V, iters)
            l1 = float(np.abs(r1.astype(np.float64) - oracle.pagerank64(og, iters, 0.85)).sum())
            assert l1 <= 1e-6, (V, iters, l1)
        g.close()


def test_automatic_layout(oracle):
    """Pairs on skewed graphs from 3 * 2^22 edges; fewer edges, no hubs: the pull."""
    m = 3 << 22
    rng = np.random.default_rng(4)
    V = 1 << 18
    for skew, e_n, layout in ((2.5, m + 600000, 5), (2.5, m - 600000, 2), (1, m + 600000, 2)):
        src = (V * rng.random(e_n) ** skew).astype(np.uint32)
        dst = rng.integers(0, V, e_n).astype(np.uint32)
        if skew > 1:
            src[:20000] = 7
        g = cg.Graph.from_edges(V, src, dst, None)
        og = oracle.csr_build(V, src, dst)
        e = cg.Engine(g, PR)
        r, st = e.run()
        e.close()
        assert st["pr_layout"] == layout, (skew, e_n, st["pr_layout"])
        assert float(np.abs(r.astype(np.float64) - oracle.pagerank64(og, 20, 0.85)).sum()) <= 1e-6
        g.close()
