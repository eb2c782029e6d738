"""Results copied out in pieces (csrc/stage.hpp): sizes around a piece and a
ring of them, memory the device reaches, two readers at once, batches sharing a
first graph."""
import ctypes
import threading

import numpy as np
import pytest
import torch

import cggraph_amd as cg
from cggraph_amd import batch

pytestmark = pytest.mark.gpu


def path(V):
    off = np.minimum(np.arange(V + 1), V - 1).astype(np.uint64)
    return cg.Graph.from_csr(off, np.arange(1, V, dtype=np.uint32))


@pytest.mark.parametrize("V", [1, 3, 2**18 - 1, 2**18, 2**18 + 1, 3 * 2**18, 3 * 2**18 + 5, 2**20 + 77])
def test_piece_sizes(V):
    off = np.zeros(V + 1, np.uint64)
    off[1:] = V - 1  # a star: vertex 0 reaches all
    g = cg.Graph.from_csr(off, np.arange(1, V, dtype=np.uint32))
    e = cg.Engine(g, 0)
    want = np.ones(V, np.uint32)
    want[0] = 0
    for _ in range(2):
        got, _ = e.run(0)
        assert np.array_equal(got, want)
    pinned = torch.empty(V, dtype=torch.int32, pin_memory=True)
    assert cg.lib().cg_engine_result(e._h, ctypes.c_void_p(pinned.data_ptr())) == 0
    assert np.array_equal(pinned.numpy().view(np.uint32), want)
    bad = []
    readers = [threading.Thread(target=lambda: [bad.append(0) for _ in range(5) if not np.array_equal(e.result(), want)])
               for _ in range(3)]
    for t in readers:
        t.start()
    for t in readers:
        t.join()
    assert not bad
    e.close()
    g.close()


def test_batches_at_once():
    a, b = path(3000), path(700)
    want = {a: np.arange(3000, dtype=np.uint32), b: np.arange(700, dtype=np.uint32)}
    bad = []

    def go():
        for _ in range(3):
            values, _ = batch.run_batch([a, b, a], [0, 0, 0], [0, 0, 0])
            bad.extend(1 for g, v in zip([a, b, a], values) if not np.array_equal(v, want[g]))

    ts = [threading.Thread(target=go) for _ in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
