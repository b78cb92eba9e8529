"""Graphs on both sides of the size up to which the host checks them (nodes and
edges together 12288) and the GPU beyond: the same faults refused with the same
messages, the graph loaded before kept, and the same network outputs from a
graph of two halves as from each half alone."""
import numpy as np
import pytest
from test_gpu_graph_checks import _faulty

from spherocyls_amd import configs, native

pytestmark = pytest.mark.gpu
LINE = 12288


def _graph(m, n):
    R, A = configs.bidisperse(n)
    s = native.System(configs.make_packing(R, A, 0.84, 9, "graph sizes"), pads=0.1)
    try:
        return m.graph_of(s)
    finally:
        s.close()


def _ring(n, e):
    """n nodes in a ring; every node of the first e - 2 n touches its second
    neighbour too, so that n + e is any even number's worth of edges."""
    pairs = {(i, (i + 1) % n) for i in range(n)}
    pairs |= {(i, (i + 2) % n) for i in range((e - 2 * n) // 2)}
    both = sorted(pairs | {(j, i) for i, j in pairs})
    recv = np.array([i for i, _ in both])
    off = np.searchsorted(recv, np.arange(n + 1)).astype(np.int32)
    rng = np.random.default_rng(n)
    return native.Graph(rng.uniform(-1, 1, (n, 4)).astype(np.float32), off,
                        np.array([j for _, j in both], np.int32),
                        rng.uniform(-1, 1, (len(both), 5)).astype(np.float32))


@pytest.mark.parametrize("kind,message", [
    ("order", "senders must increase"), ("range", "symmetric"), ("negative", "symmetric"),
    ("one way", "symmetric"), ("node", "node feature"), ("edge", "edge feature"),
    ("offsets", "offsets must not decrease")])
def test_faults_beyond_the_line(kind, message):
    m = native.Mpnn(seed=3)
    try:
        g = _graph(m, 5000)
        assert g.n + g.e > LINE
        m.load_graph(g)
        before = m.forward()
        print("large graph fault", kind, flush=True)
        with pytest.raises(native.SpherocylsError, match=message):
            m.load_graph(_faulty(g, kind))
        assert np.array_equal(m.forward(), before)
    finally:
        m.close()


@pytest.mark.parametrize("extra", [-2, 0, 2])
def test_graphs_at_the_line(extra):
    """Two copies of a graph below the line, as one graph at or beyond it."""
    m = native.Mpnn(seed=4)
    try:
        n = 1536
        g = _ring(n, LINE // 2 - n + extra // 2 * 2 if extra >= 0 else LINE // 2 - n - 2)
        two = native.Graph.concat([g, g])
        print("graph of", two.n + two.e, flush=True)
        assert g.n + g.e <= LINE and (two.n + two.e > LINE) == (extra > 0)
        m.load_graph(g)
        one = m.forward()
        m.load_graph(two)
        both = m.forward()
        assert np.array_equal(both[:n], one) and np.array_equal(both[n:], one)
        target = np.zeros((two.n, 3), np.float32)
        assert np.isfinite(m.backward(target))
    finally:
        m.close()
