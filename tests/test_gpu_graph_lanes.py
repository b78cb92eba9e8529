"""Contact graphs built by sixteen lanes a node: boxes of one, two and many rows of
cells, and a node of more contacts than the lanes order together (a large disc
among small ones).  The graph is exactly the set of touching pairs, senders in
increasing order."""
import numpy as np
import pytest

import oracle
from spherocyls_amd import configs, native

pytestmark = pytest.mark.gpu


def _packing(kind):
    rng = np.random.default_rng(23)
    if kind == "hub":  # 70 small discs touch the large one, 30 lie further out
        a = np.linspace(0, 2 * np.pi, 70, endpoint=False)
        b = np.linspace(0, 2 * np.pi, 30, endpoint=False)
        x = 12 + np.concatenate([[0], 4.1 * np.cos(a), 5.5 * np.cos(b)])
        y = 12 + np.concatenate([[0], 4.1 * np.sin(a), 5.5 * np.sin(b)])
        R = np.concatenate([[4.0], np.full(100, 0.15)])
        return configs.Packing(24.0, x, y, np.zeros(101), np.zeros(101), R, 0.0, kind)
    n, L = {"one row": (5, 4.0), "two rows": (8, 5.6), "many": (333, 30.0)}[kind]
    return configs.Packing(L, rng.uniform(0, L, n), rng.uniform(0, L, n), rng.uniform(-3, 3, n),
                           rng.uniform(0.0, 0.6, n), rng.uniform(0.4, 0.6, n), 0.0, kind)


@pytest.mark.parametrize("kind", ["one row", "two rows", "many", "hub"])
def test_graph_is_the_set_of_contacts(kind):
    pk = _packing(kind)
    print("graph lanes", kind, flush=True)
    s = native.System(pk, pads=0.1)
    m = native.Mpnn(seed=3)
    try:
        g = m.graph_of(s)
    finally:
        s.close()
        m.close()
    n = len(pk.x)
    rod = [(pk.x[i], pk.y[i], pk.phi[i], pk.A[i], pk.R[i]) for i in range(n)]
    want = [[] for _ in range(n)]
    for i in range(n):
        for j in range(i + 1, n):
            if oracle.pair_contacts(rod[i], rod[j], model=0, L=pk.L):
                want[i].append(j)
                want[j].append(i)
    if kind == "hub":
        assert len(want[0]) == 70
    got = [g.src[g.offsets[i]:g.offsets[i + 1]].tolist() for i in range(n)]
    assert got == [sorted(w) for w in want]
    assert np.all(g.edge_feat[:, 0] > 0)  # overlaps (above 1 for crossed rods)
