"""Push tiers on graphs of one vertex with most edges (csrc/kernels.hpp,
chunk_edges_for): chunks between 256 and 2048 edges, from the centre, from a
leaf, and with other rows beside it.  Bit-exact against the oracle."""
import numpy as np
import pytest

import cggraph_amd as cg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("leaves", [524_287, 524_288, 1_048_577, 2_097_153])
@pytest.mark.parametrize("sym", [False, True])
def test_star(oracle, leaves, sym):
    rng = np.random.default_rng(leaves)
    src = np.r_[np.zeros(leaves, np.int64), rng.integers(1, leaves + 1, 300_000)]
    dst = np.r_[np.arange(1, leaves + 1), rng.integers(1, leaves + 1, 300_000)]
    og = oracle.csr_build(leaves + 1, src.astype(np.uint32), dst.astype(np.uint32), symmetrize=sym)
    og.weight = rng.integers(1, 1000, og.E).astype(np.uint32)
    if sym:
        og.weight[:] = 7
    g = cg.Graph.from_csr(og.offsets, og.dest, og.weight)
    for alg in (0, 1):
        e = cg.Engine(g, alg)
        for r in (0, 5, leaves):
            got, st = e.run(r)
            ref = oracle.bfs(og, r) if alg == 0 else oracle.sssp(og, r)
            assert np.array_equal(got, ref), (alg, r)
            assert st["edges_traversed"] == oracle.reached_edges(og, ref)
        e.close()
    g.close()
