"""Label propagation with bottom-up rounds first (csrc/ccpull.hip): labels
bit-exact against the CPU oracle (smallest id among a vertex's ancestors)
where the rounds can go wrong."""
import numpy as np
import pytest

import cggraph_amd as cg
from cggraph_amd import _lib

pytestmark = pytest.mark.gpu


def check(oracle, V, src, dst, modes=(_lib.CG_SCHED_GPU, _lib.CG_SCHED_LEARNED)):
    og = oracle.csr_build(V, np.asarray(src, np.uint32), np.asarray(dst, np.uint32))
    ref = oracle.cc_directed(og)
    g = cg.Graph.from_csr(og.offsets, og.dest)
    for mode in modes:
        e = cg.Engine(g, 2, sched_mode=mode)
        for i in range(3):
            got, _ = e.run(0, copy_out=i != 1)
            assert np.array_equal(e.result() if got is None else got, ref), (V, mode, i)
        e.close()
    g.close()


@pytest.mark.parametrize("scale,ef,keep", [(13, 16, 1.0), (14, 24, 1.0), (15, 16, 0.7), (16, 9, 1.0)])
def test_skewed(oracle, scale, ef, keep):
    """R-MAT graphs; keep < 1 drops vertices' low ids from the sources, so the
    smallest source is a small vertex and the rounds may not run."""
    src, dst = oracle.rmat_edges(scale, ef, seed=scale)[:2]
    if keep < 1.0:
        ok = src >= int((1 << scale) * (1 - keep) / 8)
        src, dst = src[ok], dst[ok]
    check(oracle, 1 << scale, src, dst)


@pytest.mark.parametrize("fan", [16380, 16384, 16416, 16417, 40000])
def test_long_rows_outside_the_source(oracle, fan):
    """Vertex 0 reaches half of the graph; the other half holds a row of `fan`
    in-edges (kept to its second kernel from 16 384 + 32 on) that it does not
    reach, behind a chain that lowers the row's label several times."""
    rng = np.random.default_rng(fan)
    half = 50_000
    src = [np.zeros(half - 1, np.int64), rng.integers(1, half, 400_000)]
    dst = [np.arange(1, half), rng.integers(1, half, 400_000)]
    hub = half + fan + 20
    src += [half + 10 + np.arange(fan), [hub] * 200]
    dst += [np.full(fan, hub), hub + 1 + np.arange(200)]
    # a descending chain into one of the row's sources
    chain = [half, hub + 250, half + 3, hub + 240, half + 5, half + 10 + fan - 1]
    src.append(chain[:-1])
    dst.append(chain[1:])
    check(oracle, hub + 300, np.concatenate(src), np.concatenate(dst))


def test_row_lengths(oracle):
    """In-edge rows of 0..70 sources, most of them reached late, beside a
    vertex 0 that reaches most of the graph."""
    rng = np.random.default_rng(3)
    n = 30_000
    src, dst = [np.zeros(n - 1, np.int64), rng.integers(1, n, 90_000)], [np.arange(1, n), rng.integers(1, n, 90_000)]
    for k in range(71):
        src.append(n + rng.integers(0, 300, k))
        dst.append(np.full(k, n + 300 + k))
    src.append(n + 300 + rng.integers(0, 71, 500))
    dst.append(n + rng.integers(0, 300, 500))
    check(oracle, n + 400, np.concatenate(src), np.concatenate(dst))
