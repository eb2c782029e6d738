"""Components of symmetric graphs (csrc/wcc.hip): the first neighbour linked with
the initialisation, the second round taken or skipped by a sample.  Labels
bit-exact against the CPU oracle (the smallest vertex id of each component)."""
import numpy as np
import pytest

import cggraph_amd as cg

pytestmark = pytest.mark.gpu


def graph(oracle, V, src, dst):
    return oracle.csr_build(V, np.asarray(src, np.uint32), np.asarray(dst, np.uint32), symmetrize=True)


def cases(oracle):
    rng = np.random.default_rng(11)
    yield "lattice", oracle.grid_graph(130, 0.4, seed=4)  # many trees after round 0: second round
    yield "skewed", oracle.rmat_graph(14, 16, seed=2, symmetrize=True)  # one tree: skipped
    for V in (1, 1023, 1024, 1025):
        yield f"path {V}", graph(oracle, V, np.arange(V - 1), np.arange(1, V))
        p = rng.permutation(V)
        yield f"shuffled path {V}", graph(oracle, V, p[:-1], p[1:])
    yield "pairs", graph(oracle, 5000, np.arange(0, 5000, 2), np.arange(1, 5000, 2))
    yield "star at the end", graph(oracle, 3000, np.full(2999, 2999), np.arange(2999))
    # two halves joined by their largest ids' last edges only
    a = rng.integers(0, 2000, 9000)
    b = rng.integers(0, 2000, 9000)
    yield "two blobs", graph(oracle, 4000, np.concatenate([a, a + 2000, [1999]]), np.concatenate([b, b + 2000, [3999]]))
    yield "sparse", graph(oracle, 6000, rng.integers(0, 6000, 4000), rng.integers(0, 6000, 4000))


def test_components(oracle):
    for name, og in cases(oracle):
        ref = oracle.cc_undirected(og)
        g = cg.Graph.from_csr(og.offsets, og.dest)
        e = cg.Engine(g, 2)
        assert g.info()["symmetric"], name
        for i in range(3):
            got, st = e.run(0, copy_out=i != 1)
            assert np.array_equal(e.result() if got is None else got, ref), (name, i)
            assert st["edges_traversed"] == og.E
        e.close()
        e = cg.Engine(g, 2, profile=1)
        got, st = e.run(0)
        assert np.array_equal(got, ref) and st["expand_kernel_ms"] > 0, name
        e.close()
        g.close()
