"""PageRank row blocks (csrc/pagerank.hip) at their limits: rows around 1024
in-edges (from there on a row is cut into chunks), around 32 (a lane or half a
wavefront each), blocks filled to just below twice 1024 edges, chunk ends.
FP64 oracle; ranks are rounded to FP32 once an iteration and row sums are in
64 bits, so over 20 damped iterations the error stays below 20 * 2^-24 of the
mass of 1, with the contributions' rounding twice that: 2.4e-6 at most."""
import numpy as np
import pytest

import cggraph_amd as cg

pytestmark = pytest.mark.gpu

# in-degrees of consecutive rows; a row takes its edges + 2 of a block's 1024
ROWS = {
    "around 1024": [1022, 1023, 1024, 1025, 1026, 0, 1023, 1024, 1, 1025, 2, 2048],
    "around 32": [31, 32, 33, 0, 63, 64, 65, 1, 30] * 40,
    "full blocks": [1019, 1023, 1021, 1023, 1020, 1023] * 5,           # 2042 edges in one block
    "thirty and a long one": ([32] * 30 + [1023]) * 4,                 # 31 rows of half a wavefront each
    "lanes and a long one": ([0, 1, 2, 3] * 60 + [1023, 1024]) * 4,    # hundreds of rows in a block
    "empty rows": [0] * 2000 + [1023] + [0] * 600 + [1024, 5],
    "chunks": [4095, 4096, 4097, 8191, 8192, 8193, 1024],
}


@pytest.mark.parametrize("rows", sorted(ROWS))
def test_rows(oracle, rows):
    deg = np.array(ROWS[rows])
    V = max(len(deg), 300)
    dst = np.repeat(np.arange(len(deg)), deg)
    src = np.random.default_rng(len(deg)).integers(0, V, len(dst))
    og = oracle.csr_build(V, src.astype(np.uint32), dst.astype(np.uint32))
    g = cg.Graph.from_csr(og.offsets, og.dest)
    for layout in (1, 2):
        for iters in (1, 2, 20):
            e = cg.Engine(g, 3, pr_layout=layout, pr_iterations=iters)
            r1, _ = e.run()
            r2, _ = e.run()
            e.close()
            assert np.array_equal(r1.view(np.uint32), r2.view(np.uint32)), (layout, iters)
            l1 = float(np.abs(r1.astype(np.float64) - oracle.pagerank64(og, iters, 0.85)).sum())
            assert l1 <= 2.4e-6, (layout, iters, l1)
    g.close()
