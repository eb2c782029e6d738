"""What a level cluster (csrc/cluster.hip) leaves for the wide pipeline when it
hands a BFS frontier back: the front kernel sizes its chunk queue, chooses the
direction and adds up the traversed edges by the frontier's out-edges, so their
count has to be exact also where the cluster's report saturates (2^17 edges of
one workgroup, rows of 2^17).  Depths and traversed edges against the oracle."""
import numpy as np
import pytest

import cggraph_amd as cg

pytestmark = pytest.mark.gpu


def check(oracle, V, src, dst, roots):
    og = oracle.csr_build(V, np.concatenate(src).astype(np.uint32), np.concatenate(dst).astype(np.uint32))
    g = cg.Graph.from_csr(og.offsets, og.dest)
    e = cg.Engine(g, 0)
    for r in roots:
        ref = oracle.bfs(og, r)
        got, st = e.run(r)
        assert np.array_equal(got, ref), r
        assert st["edges_traversed"] == oracle.reached_edges(og, ref), r
    e.close()
    g.close()


# 3: the frontier is handed back as it was taken over; fewer: not the cluster's
@pytest.mark.parametrize("path", [1, 2, 3, 4, 5, 20])
@pytest.mark.parametrize("n", [300, 400, 1500])
def test_path_into_a_clique(oracle, path, n):
    """A path whose end knows a clique's first half (found by one workgroup):
    45 k, 80 k and 1.1 M out-edges in one frontier."""
    a, b = np.divmod(np.arange(n * n), n)
    c = path + np.arange(n // 2)
    check(oracle, path + n, [np.arange(path - 1), np.full(n // 2, path - 1), path + a[a != b]],
          [np.arange(1, path), c, path + b[a != b]], [0, path - 1, path, 0])


@pytest.mark.parametrize("deg", [(1 << 17) - 1, 1 << 17, 200_000])
def test_path_into_a_long_row(oracle, deg):
    """A path to a vertex whose row is as long as the report counts, its leaves
    with a vertex of their own behind each."""
    p = 12
    leaves = p + np.arange(deg)
    check(oracle, p + 2 * deg, [np.arange(p - 1), np.full(deg, p - 1), leaves],
          [np.arange(1, p), leaves, leaves + deg], [0, p - 1, 5])


@pytest.mark.parametrize("d", [6000, 8000])
def test_path_into_many_hubs(oracle, d):
    """300 hubs found by all workgroups (the 600 vertices before them are dealt
    out): with 19 hubs to a workgroup, 114 k and 152 k out-edges each."""
    p, h, mid = 8, 300, 600
    rng = np.random.default_rng(1)
    mids, hubs, leaves = p + np.arange(mid), p + mid + np.arange(h), p + mid + h
    check(oracle, leaves + 40_000, [np.arange(p - 1), np.full(mid, p - 1), mids, np.repeat(hubs, d)],
          [np.arange(1, p), mids, np.repeat(hubs, mid // h), leaves + rng.integers(0, 40_000, h * d)], [0, 3, 0])
