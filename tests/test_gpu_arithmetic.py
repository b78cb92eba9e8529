"""Corners of the arithmetic that the kernels share: angles of many turns, whose
whole turns are taken off before the sine, and a minimisation whose limit is
below the root of the smallest number."""
from decimal import Decimal, getcontext

import numpy as np
import pytest

import oracle
from spherocyls_amd import configs, native

pytestmark = pytest.mark.gpu


def _without_turns(phi):
    """phi less its whole turns, to the last bit (the oracle itself takes them
    off one by one, with a pi of 15 digits)."""
    getcontext().prec = 60
    turn = 2 * Decimal("3.14159265358979323846264338327950288419716939937510")
    exact = [Decimal(float(p)) for p in phi]
    return np.array([float(p - turn * (p / turn).to_integral_value()) for p in exact])


# The turns come off within 1e-14 of a radian (an angle of 1e12 leaves a
# remainder below 2 pi and a correction below 0.2, each rounded once), a rod's
# end moves by that, and a force by that times a few pair stiffnesses.
@pytest.mark.parametrize("angle", [2.0 ** 20 - 2.0, 2.0 ** 20, 2.0 ** 20 + 2.0, -3.0e9, 1.0e12])
def test_forces_of_rods_that_turned_often(angle):
    R, A = configs.bidisperse(130, aspect=2.0)
    pk = configs.make_packing(R, A, 0.84, 5, "many turns")
    phi = pk.phi + angle
    print("many turns", angle, flush=True)
    s = native.System(pk, pads=0.1)
    try:
        s.set_positions(pk.x, pk.y, phi)
        s.calc_se()
        fx, fy, tau = s.forces()
        phi = s.positions()[2]  # eight turns fewer: the list's sort takes them off
    finally:
        s.close()
    b = oracle.OracleBox(pk.L, pk.x, pk.y, _without_turns(phi), pk.A, pk.R, 0.1)
    b.calc_se()
    p = b.particles()
    scale = max(np.abs(p["fx"]).max(), np.abs(p["tau"]).max())
    for got, want in ((fx, p["fx"]), (fy, p["fy"]), (tau, p["tau"])):
        np.testing.assert_allclose(got, want, rtol=0, atol=1e-12 * scale)


@pytest.mark.parametrize("small", [256, 0])
def test_forceless_packing_converges_at_any_limit(small):
    """Particles out of contact have F_rms = 0, below every positive limit."""
    grid = np.arange(9) * 4.0 + 2.0
    x, y = (v.ravel() for v in np.meshgrid(grid, grid))
    pk = configs.Packing(36.0, x, y, np.zeros(81), np.full(81, 0.5), np.full(81, 0.5), 0.0, "apart")
    print("forceless", small, flush=True)
    s = native.System(pk, pads=0.1)
    try:
        s.set_small_fire(small)
        it, fr, st = s.fire(native.fire_params(ftol=1e-200))
    finally:
        s.close()
    assert st == 0 and it[0] == 0 and fr[0] == 0.0
