"""Results around the size that goes through an engine's own pinned memory
(2^16 values, csrc/stage.hpp): every algorithm, repeated reads, and engines
that are first read through device memory."""
import ctypes

import numpy as np
import pytest

import cggraph_amd as cg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [1, 65535, 65536, 65537, 2**18 + 1])
@pytest.mark.parametrize("alg", [0, 1, 2, 3])
def test_small_results(oracle, alg, V):
    rng = np.random.default_rng(V)
    og = oracle.csr_build(V, rng.integers(0, V, 2 * V).astype(np.uint32), rng.integers(0, V, 2 * V).astype(np.uint32))
    og.weight = rng.integers(1, 50, og.E).astype(np.uint32)
    g = cg.Graph.from_csr(og.offsets, og.dest, og.weight)
    e = cg.Engine(g, alg)
    for i, r in enumerate((0, V - 1, V // 2, 0)):
        got, _ = e.run(r, copy_out=i % 2 == 1)  # first runs without a copy
        p = ctypes.c_void_p()
        assert cg.lib().cg_engine_result_device(e._h, ctypes.byref(p)) == 0 and p.value
        reads = [e.result() for _ in range(4)] + ([got] if got is not None else [])
        if alg == 3:
            assert float(np.abs(reads[0].astype(np.float64) - oracle.pagerank64(og, 20, 0.85)).sum()) <= 2.4e-6
        else:
            ref = (oracle.bfs, oracle.sssp, lambda o, _: oracle.cc_directed(o))[alg](og, r)
            assert np.array_equal(reads[0], ref)
        assert all(np.array_equal(x.view(np.uint32), reads[0].view(np.uint32)) for x in reads)
    e.close()
    g.close()
