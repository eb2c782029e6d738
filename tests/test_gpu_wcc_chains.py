"""Components (csrc/wcc.hip) on graphs whose first round leaves long chains and
that are larger than one stride of the compression behind it (2^20 vertices)."""
import numpy as np
import pytest

import cggraph_amd as cg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["lattice", "path", "shuffled path"])
@pytest.mark.parametrize("V", [(1 << 20) - 1, (1 << 20) + 1, 1_700_000])
def test_long_chains(oracle, kind, V):
    if kind == "lattice":
        og = oracle.grid_graph(int(V ** 0.5) + 1, 0.3, seed=V)
    else:
        p = np.arange(V) if kind == "path" else np.random.default_rng(V).permutation(V)
        cut = np.arange(V - 1) % 1000003 != 17
        og = oracle.csr_build(V, p[:-1][cut].astype(np.uint32), p[1:][cut].astype(np.uint32), symmetrize=True)
    g = cg.Graph.from_csr(og.offsets, og.dest)
    e = cg.Engine(g, 2)
    for _ in range(2):
        assert np.array_equal(e.run(0)[0], oracle.cc_undirected(og))
    e.close()
    g.close()
