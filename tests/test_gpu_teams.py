"""Teams of workgroups (many steps in one launch) against the launches per step
they replace, which the other files compare with the oracle: sizes at the edges
of a member (one member up to 128 particles, then members of up to 64, 128 when
those are too many for the GPU), rebuilds, a remap and records inside a launch.

Both sides evaluate the same formulas; sums of at most eight contact forces and
the minimiser's sums run in another order, a difference of a few units in the
last place per step (below 1e-15 of a radius).  Over 100 steps that stays below
1e-13, and a factor of 1e4 is left for contacts that amplify it.  FP32 pair math
turns such a difference into one of FP32's last place (6e-8 of a force below 1)
in some pairs, 1e-9 of a radius per step and below 1e-7 over 100."""
import numpy as np
import pytest

from spherocyls_amd import configs, native

pytestmark = pytest.mark.gpu
TOL = {"fp64": 1e-9, "mixed": 1e-6}


def _packing(n, aspect=1.5, phi=0.80):
    R, A = configs.bidisperse(n, aspect=aspect)
    return configs.make_packing(R, A, phi, 7 + n, f"team N={n}")


def _both(pk, model, precision, run):
    out = []
    for small in (256, 0):  # teams; launches per step
        s = native.System(pk, pads=0.1)
        try:
            s.set_contact_model(model)
            s.set_precision(precision)
            s.set_small_fire(small)
            extra = run(s)
            out.append((s.positions(), s.forces(), [s.box(k) for k in range(s.npack)], extra))
        finally:
            s.close()
    return out


def _compare(a, b, sides, tol):
    for u, v in zip(a[0][:2], b[0][:2]):
        d = (u - v + 0.5 * sides) % sides - 0.5 * sides  # one side may have wrapped
        assert np.max(np.abs(d)) < tol
    d = (a[0][2] - b[0][2] + np.pi) % (2 * np.pi) - np.pi
    assert np.max(np.abs(d)) < tol
    for u, v in zip(a[1], b[1]):
        assert np.max(np.abs(u - v)) < tol * max(1.0, np.max(np.abs(v)))
    for p, q in zip(a[2], b[2]):
        assert p["iters"] == q["iters"]
        assert abs(p["gamma"] - q["gamma"]) < 1e-14
        assert abs(p["gamma_total"] - q["gamma_total"]) < 1e-13


@pytest.mark.parametrize("n,model,precision", [
    (63, "two_point", "fp64"), (65, "closest", "mixed"), (128, "two_point", "mixed"),
    (129, "closest", "fp64"), (1000, "two_point", "mixed"), (33000, "two_point", "fp64"),
    ((65, 700, 129), "two_point", "fp64")])
def test_minimisers(n, model, precision):
    """30 FIRE iterations and 30 gradient-descent steps (with rebuilds) end in
    the same state; of several packings in one launch too."""
    sizes = n if isinstance(n, tuple) else (n,)
    pk = [_packing(m, phi=0.84) for m in sizes]
    sides = np.concatenate([np.full(p.x.size, p.L) for p in pk])
    params = native.fire_params(dt0=0.05, dt_max=0.5, max_move=0.02, ftol=1e-12, max_iter=30)
    print("team minimisers", n, model, precision, flush=True)
    a, b = _both(pk, model, precision, lambda s: s.fire(params, check=False)[0].tolist())
    assert a[3] == b[3]
    _compare(a, b, sides, TOL[precision])
    a, b = _both(pk, model, precision, lambda s: s.gd_steps(30))
    assert a[3] == b[3]
    _compare(a, b, sides, TOL[precision])


@pytest.mark.parametrize("n,model,precision,every,step", [
    (64, "closest", "fp64", 0, 0.02), (128, "two_point", "fp64", 7, 0.02),
    (129, "two_point", "mixed", 0, 0.02), (700, "closest", "fp64", 50, 0.02),
    (700, "closest", "mixed", 50, 0.02), (33000, "closest", "fp64", 13, 0.02),
    (700, "closest", "fp64", 0, 0.5)])
def test_sheared_steps(n, model, precision, every, step):
    """100 steps that pass the remap strain and several list windows, with
    stress records.  With steps of 0.5 particles move more than half the skin in
    a step, which a team gives up, unwritten, for the launches per step."""
    pk = _packing(n)
    print("team shear", n, model, precision, every, step, flush=True)

    def run(s):
        s.set_dynamics(strain_rate=5e-4 / step, step=step)
        s.set_gamma(0.48, 0.48)
        return s.strain_steps(100, every)

    a, b = _both(pk, model, precision, run)
    assert b[2][0]["gamma"] < 0.0  # remapped
    _compare(a, b, pk.L, TOL[precision])
    assert a[3].shape == b[3].shape
    scale = np.abs(b[3]).max() if b[3].size else 1.0
    np.testing.assert_allclose(a[3], b[3], rtol=0, atol=TOL[precision] * scale)
