"""Level cluster (csrc/cluster.hip): rows around an entry's 64 edges and
frontiers around the 1024 entries that a workgroup holds in LDS and the 8192
altogether, on an engine and in a batch.  Bit-exact against the oracle."""
import numpy as np
import pytest

import cggraph_amd as cg
from cggraph_amd import batch

pytestmark = pytest.mark.gpu
BFS, SSSP, CC = 0, 1, 2


@pytest.mark.parametrize("deg", [1, 63, 64, 65, 127, 128, 129, 1023, 1024, 1025, 8191, 8192, 8193])
def test_rows_and_queues(oracle, deg):
    """A path to a row of deg leaves, a vertex behind each leaf, all of those
    into one, and a path from there."""
    p = 6
    a, b, end = p + np.arange(deg), p + deg + np.arange(deg), p + 2 * deg
    src = np.concatenate([np.arange(p - 1), np.full(deg, p - 1), a, b, end + np.arange(p)])
    dst = np.concatenate([np.arange(1, p), a, b, np.full(deg, end), end + 1 + np.arange(p)])
    og = oracle.csr_build(end + p + 1, src.astype(np.uint32), dst.astype(np.uint32))
    og.weight = np.random.default_rng(deg).integers(1, 100, og.E).astype(np.uint32)
    roots = [0, p - 1, p, end]
    h = cg.Graph.from_csr(og.offsets, og.dest, og.weight)
    ref = {BFS: oracle.bfs, SSSP: oracle.sssp, CC: lambda g, r: oracle.cc_directed(g)}
    for alg, opt in ((BFS, {}), (SSSP, {}), (SSSP, {"sssp_delta": 60}), (CC, {})):
        e = cg.Engine(h, alg, **opt)
        for r in roots:
            assert np.array_equal(e.run(r)[0], ref[alg](og, r)), (alg, r, opt)
        e.close()
    for delta in (0, 60):
        outs, _ = batch.run_batch([h] * 8, [BFS] * 4 + [SSSP] * 4, roots * 2, sssp_delta=delta)
        for i, got in enumerate(outs):
            assert np.array_equal(got, ref[i // 4](og, roots[i % 4])), (i, delta)
    h.close()
