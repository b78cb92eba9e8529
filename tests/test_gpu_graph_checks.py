"""A graph handed to the network is checked on the GPU: every fault is refused
with its own message, and the graph loaded before stays."""
import copy

import numpy as np
import pytest

from spherocyls_amd import configs, native

pytestmark = pytest.mark.gpu


def _faulty(g, kind):
    b = copy.copy(g)
    b.offsets, b.src = g.offsets.copy(), g.src.copy()
    b.node_feat, b.edge_feat = g.node_feat.copy(), g.edge_feat.copy()
    deg = np.diff(g.offsets)
    i = int(np.flatnonzero(deg >= 2)[-1])  # a late receiver with two edges
    k = int(g.offsets[i])
    if kind == "order":
        b.src[k], b.src[k + 1] = b.src[k + 1], b.src[k]
    elif kind == "range":
        b.src[g.offsets[i + 1] - 1] = g.n
    elif kind == "negative":
        b.src[k] = -1
    elif kind == "one way":
        # the last sender of a receiver replaced by a higher one it does not touch
        last = int(g.offsets[i + 1]) - 1
        free = [j for j in range(int(g.src[last]) + 1, g.n)
                if j != i and i not in g.src[g.offsets[j]:g.offsets[j + 1]]]
        b.src[last] = free[0]
    elif kind == "node":
        b.node_feat[g.n - 1, 3] = np.nan
    elif kind == "edge":
        b.edge_feat[g.e - 1, 4] = -np.inf
    elif kind == "offsets":
        b.offsets[1] = -1
    return b


@pytest.mark.parametrize("kind,message", [
    ("order", "senders must increase"), ("range", "symmetric"), ("negative", "symmetric"),
    ("one way", "symmetric"), ("node", "node feature"), ("edge", "edge feature"),
    ("offsets", "offsets must not decrease")])
def test_faulty_graphs_are_refused(kind, message):
    R, A = configs.bidisperse(260)
    s = native.System(configs.make_packing(R, A, 0.84, 9, "graph checks"), pads=0.1)
    m = native.Mpnn(seed=3)
    try:
        g = m.graph_of(s)
        m.load_graph(g)
        before = m.forward()
        print("graph fault", kind, flush=True)
        with pytest.raises(native.SpherocylsError, match=message):
            m.load_graph(_faulty(g, kind))
        assert np.array_equal(m.forward(), before)
        m.load_graph(g)
        assert np.array_equal(m.forward(), before)
    finally:
        s.close()
        m.close()
