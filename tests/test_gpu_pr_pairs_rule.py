"""The automatic PageRank layout from 2^22 vertices on: pairs on graphs of few
(source, bin) pairs or a hot destination bin, the blocked layout where one hub
or skewed sources alone leave a pair for almost every edge.  FP64 oracle; both
layouts round contributions to FP32 and sum in 64-bit fixed point, so twenty
damped iterations stay below 2.4e-6 of the mass of 1."""
import numpy as np
import pytest

import cggraph_amd as cg

pytestmark = pytest.mark.gpu
V, M = 1 << 22, 3 << 22


def edges(kind):
    rng = np.random.default_rng(8)
    m = M + 400_000
    s, d = rng.integers(0, V, m), rng.integers(0, V, m)
    if kind == "one hub":
        s[:100] = 7
    elif kind != "uniform":
        s = (V * rng.random(m) ** 3).astype(np.int64)  # sources skewed, destinations not
        if kind == "hot bins":
            d = (V * rng.random(m) ** 3).astype(np.int64)
        elif kind == "few pairs":
            d = s // 4 + rng.integers(0, V // 512, m)
    return s.astype(np.uint32), d.astype(np.uint32)


@pytest.mark.parametrize("kind,layout", [("uniform", 4), ("one hub", 4), ("sources", 4), ("hot bins", 5), ("few pairs", 5)])
def test_layout(oracle, kind, layout):
    s, d = edges(kind)
    og = oracle.csr_build(V, s, d)
    g = cg.Graph.from_csr(og.offsets, og.dest)
    assert np.diff(og.offsets.astype(np.int64)).max() >= (16 * 4 if kind != "uniform" else 0)
    e = cg.Engine(g, 3)
    r, st = e.run()
    assert st["pr_layout"] == layout
    assert float(np.abs(r.astype(np.float64) - oracle.pagerank64(og, 20, 0.85)).sum()) <= 2.4e-6
    e.close()
    e = cg.Engine(g, 3, pr_layout=5)  # asked for, it is built whatever the rule says
    assert e.run()[1]["pr_layout"] == 5
    e.close()
    g.close()
