"""Resize steps keep a particle's row while the box changes.  The tile path has
no rows: its passes look through the cells of every state, so it is the
reference.  Both evaluate the same formulas and differ in the order of sums
(1e-15 of a radius per step, as 1e-13 over 100 steps, with a factor of 1e4 left
for contacts that amplify it)."""
import numpy as np
import pytest

from spherocyls_amd import configs, native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,phi,rate,shrink,corrected", [
    (130, 0.60, 2e-3, True, True),   # 10% in 50 steps: rows age by the shrinking alone
    (130, 0.84, 2e-3, False, True),  # growing: only the particles' own moves count
    (130, 0.84, 1e-4, True, False),  # images of the old box on positions of the new
    (2500, 0.80, 1e-3, True, False),
    (2500, 0.50, 5e-3, True, True)])
def test_rows_kept_over_box_changes(n, phi, rate, shrink, corrected):
    R, A = configs.bidisperse(n, aspect=1.5)
    pk = configs.make_packing(R, A, phi, 3 + n, f"resize N={n}")
    out = []
    for path in ("list", "tile"):
        print("resize rows", n, phi, rate, shrink, corrected, path, flush=True)
        s = native.System(pk, pads=0.1)
        try:
            s.set_path(path)
            s.set_dynamics(resize_rate=rate / 0.02, step=0.02)
            s.resize_steps(50, shrink=shrink, corrected_image=corrected)
            s.set_dynamics(strain_rate=0.01, step=0.02)
            s.strain_steps(10)  # rows of the resize passes do not outlive them
            out.append((s.positions(), s.forces(), s.box(0)))
        finally:
            s.close()
    (pa, fa, ba), (pb, fb, bb) = out
    assert ba["Lx"] == bb["Lx"] and ba["Ly"] == bb["Ly"] and ba["ncontacts"] == bb["ncontacts"]
    assert abs(ba["Lx"] / pk.L - (1 - rate / 0.02) ** ((0.02 if shrink else -0.02) * 50)) < 1e-12
    for u, v, L in zip(pa, pb, (ba["Lx"], ba["Ly"], 2 * np.pi)):
        d = u - v
        assert np.max(np.abs(d - L * np.round(d / L))) < 1e-9
    for u, v in zip(fa, fb):
        assert np.max(np.abs(u - v)) < 1e-9 * max(1.0, np.max(np.abs(v)))
