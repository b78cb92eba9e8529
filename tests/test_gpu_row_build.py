"""Rows built by the lanes of a particle together: grids of one, two and three
rows of cells, buckets up to every sorting width and beyond the widest (crowded
cells of a polydisperse packing), each number of lanes.  Forces against the
oracle: sums of at most 40 contacts, each right to a few units in the last
place, so within 1e-12 of the largest force."""
import numpy as np
import pytest

import oracle
from spherocyls_amd import configs, native

pytestmark = pytest.mark.gpu


def _packing(kind):
    rng = np.random.default_rng(17)
    if kind == "crowded":  # small rods among a few large ones: some 40 to a cell
        n, L = 400, 14.0
        R = np.where(np.arange(n) % 50 == 0, 0.8, rng.uniform(0.08, 0.16, n))
        A = 0.5 * R
    else:
        n, L = {"one cell": (5, 4.0), "two rows": (8, 5.6), "three rows": (26, 9.8),
                "many": (700, 44.0)}[kind]
        R = rng.uniform(0.4, 0.6, n)
        A = rng.uniform(0.0, 0.6, n)
    x, y = rng.uniform(0, L, n), rng.uniform(0, L, n)
    return configs.Packing(L, x, y, rng.uniform(-3, 3, n), A, R, 0.0, kind)


def _reference(pk, kind):
    """Forces and contacts.  (The oracle's box visits a cell of a grid of fewer
    than three rows more than once, so those are summed pair by pair.)"""
    if kind not in ("one cell", "two rows"):
        b = oracle.OracleBox.from_packing(pk, 0.1)
        b.calc_se()
        p = b.particles()
        return np.array([p["fx"], p["fy"], p["tau"]]), len(b.brute_contacts()[0])
    n, f, contacts = len(pk.x), np.zeros((3, len(pk.x))), 0
    rod = [(pk.x[i], pk.y[i], pk.phi[i], pk.A[i], pk.R[i]) for i in range(n)]
    for i in range(n):
        for j in range(i + 1, n):
            for c in oracle.pair_contacts(rod[i], rod[j], model=0, L=pk.L):
                contacts += 1
                f[:, i] += c["fx"], c["fy"], c["tau_p"]
                f[:, j] += -c["fx"], -c["fy"], c["tau_q"]
    return f, contacts


@pytest.mark.parametrize("kind", ["one cell", "two rows", "three rows", "many", "crowded"])
@pytest.mark.parametrize("lanes", [1, 2, 4, 8])
def test_forces_on_rebuilt_rows(kind, lanes):
    pk = _packing(kind)
    print("row build", kind, lanes, flush=True)
    s = native.System(pk, pads=0.1)
    try:
        s.set_path("list")
        s.set_list_block(128, lanes)
        s.set_positions(pk.x, pk.y, pk.phi)  # (a rebuild)
        s.calc_se()
        got = s.forces()
        box = s.box()
    finally:
        s.close()
    want, contacts = _reference(pk, kind)
    scale = np.abs(want).max()
    assert scale > 0
    for u, v in zip(got, want):
        np.testing.assert_allclose(u, v, rtol=0, atol=1e-12 * scale)
    assert box["ncontacts"] == contacts
