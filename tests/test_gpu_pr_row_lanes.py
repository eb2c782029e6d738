"""PageRank with a lane or a wavefront a row (csrc/pagerank.hip), on either side
of the rule that takes them: longest row 1, 2, 3, 6, 7, rows of about 384 in-edges
and unlike ones, up to and past 2^19 rows, in the caller's order and renumbered.
FP64 oracle, bound as derived in test_gpu_pr_row_limits.py."""
import numpy as np
import pytest

import cggraph_amd as cg

pytestmark = pytest.mark.gpu


def check(oracle, V, src, dst, layouts=(1, 2)):
    og = oracle.csr_build(V, src.astype(np.uint32), dst.astype(np.uint32))
    g = cg.Graph.from_csr(og.offsets, og.dest)
    for layout in layouts:
        for iters in (1, 2, 20):
            e = cg.Engine(g, 3, pr_layout=layout, pr_iterations=iters)
            r1, _ = e.run()
            assert np.array_equal(e.run()[0].view(np.uint32), r1.view(np.uint32))
            e.close()
            assert float(np.abs(r1.astype(np.float64) - oracle.pagerank64(og, iters, 0.85)).sum()) <= 2.4e-6
    g.close()


@pytest.mark.parametrize("longest", [1, 2, 3, 6, 7])
@pytest.mark.parametrize("V", [1, 255, 257, 5000, 2**19 - 1, 2**19, 2**19 + 1])
def test_short_rows(oracle, longest, V):
    rng = np.random.default_rng(V + longest)
    deg = rng.integers(0, longest + 1, V)
    deg[V // 2] = longest
    dst = np.repeat(np.arange(V), deg)
    check(oracle, V, rng.integers(0, V, len(dst)), dst)


@pytest.mark.parametrize("V", [1, 63, 700])
@pytest.mark.parametrize("deg", [(383, 383), (384, 384), (385, 700), (384, 900), (1023, 1025), (4096, 4097)])
def test_long_rows(oracle, V, deg):
    """All rows as long as the first, but the last: the second."""
    d = np.full(V, deg[0])
    d[-1] = deg[1]
    dst = np.repeat(np.arange(V), d)
    check(oracle, V, np.random.default_rng(V).integers(0, V, len(dst)), dst)
