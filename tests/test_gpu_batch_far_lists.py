"""Bucketed SSSP of a batch on level clusters when more vertices wait than the
far lists have room for (8192 a workgroup): they wait in a bitmap instead, for
one bucket or for many, are dropped once their value has improved, and the
buckets stay what they are.  Bit-exact against the oracle."""
import numpy as np
import pytest

import cggraph_amd as cg
from cggraph_amd import batch

pytestmark = pytest.mark.gpu


def csr(oracle, V, src, dst, w):
    og = oracle.csr_build(V, np.concatenate(src).astype(np.uint32), np.concatenate(dst).astype(np.uint32))
    og.weight = w(og.E).astype(np.uint32)
    return og


def fan(oracle, lo, hi):
    """A root that reaches 192 000 leaves in three steps of at most 64 edges, each
    with a vertex of its own behind it and a short cut from another leaf, so
    that half of the waiting values improve while they wait."""
    rng = np.random.default_rng(hi)
    mid, n = 5000, 192_000
    leaves = mid + np.arange(n)
    src = [np.zeros(50, np.int64), np.repeat(np.arange(1, 51), 60), np.repeat(np.arange(51, 3051), 64), leaves, leaves]
    dst = [np.arange(1, 51), np.arange(51, 3051), leaves, leaves + n, mid + rng.integers(0, n, n)]
    return csr(oracle, mid + 2 * n, src, dst, lambda E: rng.integers(lo, hi, E))


def lattice3(oracle, n):
    i = np.arange(n ** 3)
    src, dst = [], []
    for c, step in ((i % n, 1), (i // n % n, n), (i // n ** 2, n * n)):
        k = i[c < n - 1]
        src += [k, k + step]
        dst += [k + step, k]
    return csr(oracle, n ** 3, src, dst, lambda E: np.random.default_rng(n).integers(1, 1001, E))


# 2: 16 workgroups to a cluster (131 072 entries), 40: 4 (32 768)
@pytest.mark.parametrize("queries", [2, 40])
@pytest.mark.parametrize("delta", [50, 1000, 30_000, 4_000_000_000])
def test_waiting_vertices_beyond_the_lists(oracle, queries, delta):
    graphs = [fan(oracle, 40, 60_000), fan(oracle, 900, 1100), lattice3(oracle, 66)]
    handles = [cg.Graph.from_csr(o.offsets, o.dest, o.weight) for o in graphs]
    roots = [[0, 60], [0, 5000], [0, 66 ** 3 // 2]]
    refs = [[oracle.sssp(o, r) for r in rs] for o, rs in zip(graphs, roots)]
    assert all(np.diff(o.offsets.astype(np.int64)).max() <= 64 for o in graphs)
    for k in range(3):
        qs = [(k, i % 2) for i in range(queries)]
        outs, st = batch.run_batch([handles[k]] * queries, [1] * queries, [roots[k][i] for _, i in qs], sssp_delta=delta)
        for (_, i), got in zip(qs, outs):
            assert np.array_equal(got, refs[k][i]), (k, i)
        assert st["edges_traversed"] == sum(oracle.reached_edges(graphs[k], refs[k][i]) for _, i in qs)
    for h in handles:
        h.close()
