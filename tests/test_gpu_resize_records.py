"""Stress records inside resize runs: their force passes use the rows kept over
the box changes.  The tile path has no rows and is the reference (as for the
trajectories in test_gpu_resize_rows); sums run in another order, 1e-13 over 60
steps with a factor of 1e4 left for contacts that amplify it."""
import numpy as np
import pytest

from spherocyls_amd import configs, native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,phi,rate,shrink,corrected,every", [
    (130, 0.80, 2e-3, True, True, 1),
    (130, 0.84, 2e-3, False, True, 7),
    (900, 0.84, 2e-4, True, False, 3),
    (2500, 0.80, 1e-3, True, True, 20)])
def test_records_of_a_resize_run(n, phi, rate, shrink, corrected, every):
    R, A = configs.bidisperse(n, aspect=1.5)
    pk = configs.make_packing(R, A, phi, 5 + n, f"resize records N={n}")
    out = []
    for path in ("list", "tile"):
        print("resize records", n, rate, shrink, path, flush=True)
        s = native.System(pk, pads=0.1)
        try:
            s.set_path(path)
            s.set_dynamics(resize_rate=rate / 0.02, step=0.02)
            out.append(s.resize_steps(60, shrink=shrink, corrected_image=corrected,
                                      se_every=every))
        finally:
            s.close()
    a, b = out
    assert a.shape == b.shape == (60 // every, 1, 9)
    np.testing.assert_array_equal(a[..., 8], b[..., 8])  # contacts
    np.testing.assert_allclose(a, b, rtol=0, atol=1e-9 * np.abs(b[..., :8]).max())
