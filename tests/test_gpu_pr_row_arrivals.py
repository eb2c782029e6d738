"""PageRank rows cut into chunks that end on any workgroup (csrc/pagerank.hip):
hundreds of rows of several chunks each, every run bit-identical.  FP64 oracle,
bound as derived in test_gpu_pr_row_limits.py."""
import numpy as np
import pytest

import cggraph_amd as cg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,deg", [(600, 9000), (40, 200_000), (3, 1_500_001)])
def test_many_chunks(oracle, rows, deg):
    V = 60_000
    rng = np.random.default_rng(rows)
    dst = np.repeat(rng.choice(V, rows, replace=False), deg)
    src = rng.integers(0, V, len(dst))
    og = oracle.csr_build(V, src.astype(np.uint32), dst.astype(np.uint32))
    g = cg.Graph.from_csr(og.offsets, og.dest)
    ref = oracle.pagerank64(og, 20, 0.85)
    e = cg.Engine(g, 3, pr_layout=1)
    first, _ = e.run()
    assert float(np.abs(first.astype(np.float64) - ref).sum()) <= 2.4e-6
    for _ in range(4):
        assert np.array_equal(e.run()[0].view(np.uint32), first.view(np.uint32))
    e.close()
    g.close()
