"""Which calls run as teams of workgroups, and what a team does where it cannot
go on: the launch counter and its status say so, and the steps are compared with
the launches per step (whose results the other files compare with the oracle).

A member of a team holds 64 particles and at most 448 around them.  With a few
large discs the cells are large, and a member's cells hold more particles than
that, at once or once its own have drifted over more cells; _halo computes the
count.  Both sides evaluate the same formulas and differ in the order of sums (a
few units in the last place per step, as 1e-13 over 150, with a factor of 1e4
left for contacts that amplify it)."""
import numpy as np
import pytest

from spherocyls_amd import configs, native

pytestmark = pytest.mark.gpu
ROOM = 448
TOL = 1e-9


def _packing(n, seed, discs=0, radius=0.0, phi=0.84):
    R, A = configs.bidisperse(n, aspect=1.5)
    R[:discs], A[:discs] = radius, 0.0
    return configs.make_packing(R, A, phi, seed, f"N={n} with {discs} discs")


def _cells(pk, x, y):
    g = int(pk.L / (2 * (pk.R.max() + pk.A.max()) + 0.1))
    return g, (y % pk.L * (g / pk.L)).astype(int) % g, (x % pk.L * (g / pk.L)).astype(int) % g


def _halo(pk, x, y):
    """Most particles around a member, of members that hold runs of the
    packing's storage order (by cell and number at its start)."""
    g, r0, c0 = _cells(pk, pk.x, pk.y)
    order = np.lexsort((np.arange(pk.n), r0 * g + c0))
    _, r, c = _cells(pk, x, y)
    per = -(-pk.n // -(-pk.n // 64))
    most = 0
    for at in range(0, pk.n, per):
        own, near = order[at:at + per], np.zeros((g, g), bool)
        for d in (-1, 0, 1):
            for e in (-1, 0, 1):
                near[(r[own] + d) % g, (c[own] + e) % g] = True
        most = max(most, int(near[r, c].sum()) - len(own))
    return most


def _system(pk, small):
    s = native.System(pk, pads=0.1)
    s.set_contact_model("two_point")
    s.set_small_fire(small)
    return s


def _same(a, b, L, tol=TOL):
    for u, v, side in zip(a[0], b[0], (L, L, 2 * np.pi)):
        d = u - v
        assert np.max(np.abs(d - side * np.round(d / side))) < tol
    for u, v in zip(a[1], b[1]):
        assert np.max(np.abs(u - v)) < tol * max(1.0, np.max(np.abs(v)))


@pytest.mark.parametrize("n", [100, 700, 16384])
def test_calls_that_run_as_teams(n):
    pk = _packing(n, 3, phi=0.80)
    s = _system(pk, 256)
    try:
        print("teams", n, flush=True)
        s.fire(native.fire_params(max_move=0.02, ftol=1e-12, max_iter=200), check=False)
        assert s.team_info() == (1, 0)
        s.gd_steps(30)
        assert s.team_info() == (2, 0)
        s.set_dynamics(strain_rate=1e-3, step=0.005)
        s.strain_steps(100)
        assert s.team_info() == (3, 0)
        s.strain_steps(100, 20)
        assert s.team_info() == (4, 0)
        s.set_small_fire(0)
        s.strain_steps(100)
        s.gd_steps(5)
        assert s.team_info() == (4, 0)
    finally:
        s.close()


def test_no_room_while_minimising():
    """FIRE and gradient descent whose members run out of room on the way: the
    state reached goes on with the launches per step."""
    pk = _packing(1000, 1, discs=2, radius=3.0)
    assert _halo(pk, pk.x, pk.y) <= ROOM  # a team starts
    params = native.fire_params(dt0=0.05, dt_max=0.5, max_move=0.02, ftol=1e-12, max_iter=60)
    for name, run in (("fire", lambda s: s.fire(params, check=False)[0][0]),
                      ("descent", lambda s: s.gd_steps(60))):
        out = []
        for small in (256, 0):
            print("no room,", name, small, flush=True)
            s = _system(pk, small)
            try:
                s.set_dynamics(step=0.05)
                assert run(s) == 60
                assert s.team_info() == ((1, native.SC_TEAM_NO_ROOM) if small else (0, 0))
                out.append((s.positions(), s.forces()))
            finally:
                s.close()
        assert _halo(pk, *out[1][0][:2]) > ROOM
        _same(*out, pk.L)


def test_no_room_during_sheared_steps_with_records():
    pk = _packing(1000, 1, discs=2, radius=3.0)
    assert _halo(pk, pk.x, pk.y) <= ROOM
    out = []
    for small in (256, 0):
        print("no room, shear", small, flush=True)
        s = _system(pk, small)
        try:
            s.set_dynamics(strain_rate=1e-3, step=0.004)
            se = s.strain_steps(150, 7)
            assert s.team_info() == ((1, native.SC_TEAM_NO_ROOM) if small else (0, 0))
            out.append((s.positions(), s.forces(), se, s.box(0)))
        finally:
            s.close()
    assert _halo(pk, *out[1][0][:2]) > ROOM
    _same(out[0], out[1], pk.L)
    assert out[0][2].shape == (21, 1, 9)
    np.testing.assert_allclose(out[0][2], out[1][2], rtol=0, atol=TOL * np.abs(out[1][2]).max())
    assert out[0][3]["gamma"] == pytest.approx(out[1][3]["gamma"], abs=1e-14)


def test_outrun_rows():
    """Steps in which particles move more than half the skin."""
    pk = _packing(700, 5, phi=0.80)
    out = []
    for small in (256, 0):
        print("outrun", small, flush=True)
        s = _system(pk, small)
        try:
            s.set_dynamics(strain_rate=1e-3, step=0.5)
            s.strain_steps(100)
            assert s.team_info() == ((1, native.SC_TEAM_OUTRAN) if small else (0, 0))
            out.append((s.positions(), s.forces()))
        finally:
            s.close()
    _same(*out, pk.L)


def test_launches_go_on_after_a_team_in_the_middle():
    """A batch too large for teams, whose loose packings finish at once: the
    rest go on as teams, which have no room from their first pass on, and then
    with the launches per step again.  (The sheared step before turns the
    bucket buffers, so that the launches before and after the team read
    different ones.)"""
    tight = _packing(1000, 1, discs=2, radius=4.0)
    at = np.arange(1000)  # on a lattice, out of reach of each other
    loose = configs.Packing(80.0, 2.5 * (at % 32) + 1.0, 2.5 * (at // 32) + 1.0, 0.1 * at,
                            0.5 * np.ones(1000), 0.5 * np.ones(1000), 0.0, "loose")
    assert _halo(tight, tight.x, tight.y) > ROOM
    packs = [tight if k % 8 < 3 else loose for k in range(80)]  # 30 tight
    params = native.fire_params(dt0=0.05, dt_max=0.5, max_move=0.02, ftol=1e-12, max_iter=120)
    out = []
    for small in (256, 0):
        print("team in the middle", small, flush=True)
        s = _system(packs, small)
        try:
            s.set_dynamics(strain_rate=1e-4, step=0.001)
            s.strain_steps(1)
            it, fr, _ = s.fire(params, check=False)
            assert s.team_info() == ((1, native.SC_TEAM_NO_ROOM) if small else (0, 0))
            out.append((s.positions(), s.forces(), it, fr))
        finally:
            s.close()
    np.testing.assert_array_equal(out[0][2], out[1][2])
    assert sorted(set(out[0][2].tolist())) == [0, 120]
    np.testing.assert_allclose(out[0][3], out[1][3], rtol=1e-6)
    side = np.concatenate([np.full(p.n, p.L) for p in packs])
    _same(out[0], out[1], side)


def test_a_roll_call_in_vain():
    """With no time to wait for each other, 256 workgroups leave at once and
    unwritten (they do not come up within one look of the first): the calls give
    what the launches per step give, bit for bit, and the next ones don't try."""
    pk = _packing(16384, 4, phi=0.80)
    params = native.fire_params(dt0=0.05, dt_max=0.5, max_move=0.02, ftol=1e-12, max_iter=20)
    out = []
    for small in (256, 0):
        s = _system(pk, small)
        try:
            for name, run in (("fire", lambda: s.fire(params, check=False)),
                              ("descent", lambda: s.gd_steps(20)),
                              ("shear", lambda: s.strain_steps(40, 10))):
                print("roll call,", name, small, flush=True)
                s.set_positions(pk.x, pk.y, pk.phi)
                s.set_dynamics(strain_rate=1e-3, step=0.005)
                s.set_team_wait(0.0)
                n = s.team_info()[0]
                run()
                got = [np.concatenate([*s.positions(), *s.forces()])]
                if small:
                    assert s.team_info() == (n + 1, native.SC_TEAM_ABSENT)
                run()
                got.append(np.concatenate([*s.positions(), *s.forces()]))
                if small:
                    assert s.team_info() == (n + 1, native.SC_TEAM_ABSENT)
                out.append(got)
            s.set_team_wait(0.2)
            s.gd_steps(5)
            assert s.team_info() == ((4, 0) if small else (0, 0))
            for bad in (-0.1, 5.1, float("nan")):
                with pytest.raises(native.SpherocylsError):
                    s.set_team_wait(bad)
        finally:
            s.close()
    for a, b in zip(out[:3], out[3:]):
        for u, v in zip(a, b):
            np.testing.assert_array_equal(u, v)


@pytest.mark.parametrize("n", [60, 128, 200, 700])
def test_scalars_of_a_run_that_ends_non_finite(n):
    """The first iteration raises the time step without bound and moves
    particles out of the numbers; the run ends there, and the scalars are those
    after that iteration, as the positions are."""
    s = _system(_packing(n, 6), 256)
    try:
        print("non-finite", n, flush=True)
        p = native.fire_params(dt0=0.01, dt_max=1e300, n_min=0, f_inc=1e200, max_move=0.02)
        with pytest.raises(native.SpherocylsError, match="non-finite"):
            s.fire(p)
        assert s.team_info() == (1, 0)
        b = s.box(0)
        assert b["fire_dt"] == pytest.approx(1e198) and b["fire_alpha"] == pytest.approx(0.099)
    finally:
        s.close()


@pytest.mark.parametrize("n,rate,gamma,every", [
    (512, 0.04, 0.0, 3), (512, 0.04, 0.3, 4), (4096, 0.03, 0.2, 1), (4096, 0.04, 0.24, 2),
    (16384, 0.04, 0.0, 5), (16384, 0.03, 0.3, 0)])
def test_steps_before_one_that_outran_the_rows_stay(n, rate, gamma, every):
    """A relaxed packing sheared so fast that overlaps and speeds grow: the
    launches per step go on from the last step whose rows held, with its strain
    (before or across the remap at 0.5) and records."""
    pk = _packing(n, 8, phi=0.84)
    params = native.fire_params(dt0=0.05, dt_max=0.5, max_move=0.02, ftol=1e-9, max_iter=400)
    steps, out = 24, []
    for small in (256, 0):
        print("outrun on the way", n, rate, gamma, small, flush=True)
        s = _system(pk, 0)
        try:
            s.set_gamma(gamma, gamma)
            s.fire(params, check=False)
            s.set_small_fire(small)
            s.set_dynamics(strain_rate=rate / 0.4, step=0.4)
            se = s.strain_steps(steps, every)
            if small:
                print("steps of the team", s.team_steps(), flush=True)
                assert s.team_info() == (1, native.SC_TEAM_OUTRAN)
                assert 0 < s.team_steps() < steps
            out.append((s.positions(), s.forces(), se, s.box(0)))
        finally:
            s.close()
    _same(out[0], out[1], pk.L)
    if every:
        scale = np.abs(out[1][2]).max()
        np.testing.assert_allclose(out[0][2], out[1][2], rtol=0, atol=TOL * scale)
    for key in ("gamma", "gamma_total"):
        assert out[0][3][key] == pytest.approx(out[1][3][key], abs=1e-13)


@pytest.mark.parametrize("n,least", [(100, 8), (700, 8), (16384, 14), (60001, 32)])
def test_short_sheared_calls_are_launched_step_by_step(n, least):
    """A team's coming and going costs more than the first few steps save; calls
    below the line are the launches per step, bit for bit."""
    pk = _packing(n, 9, phi=0.7)
    out = []
    for small in (256, 0):
        s = _system(pk, small)
        try:
            print("short", n, small, flush=True)
            s.set_dynamics(strain_rate=1e-3, step=0.002)
            for k in (1, 2, least - 1):
                s.strain_steps(k, 2)
            assert s.team_info() == (0, 0)
            out.append((s.positions(), s.forces()))
            s.strain_steps(least)
            assert s.team_info()[0] == (1 if small else 0)
        finally:
            s.close()
    for a, b in zip(*out):
        for u, v in zip(a, b):
            np.testing.assert_array_equal(u, v)


@pytest.mark.parametrize("n", [128, 4096])
def test_autotuner_keeps_the_path_of_teams(n):
    """At these sizes a pass of the tile path is the fastest, but a team's
    sheared step takes less than either path's two passes."""
    s = _system(_packing(n, 5, phi=0.80), 256)
    try:
        print("autotune", n, flush=True)
        assert s.autotune(reps=3)["path"] == "list"
        s.set_dynamics(strain_rate=1e-3, step=0.005)
        s.strain_steps(50)
        assert s.team_info()[0] == 1
    finally:
        s.close()


def test_fire_autotuner_tries_shapes_by_launches():
    """Of the trials (two rounds) only the team's own are team launches; the
    setting outlives them, also where a trial fails."""
    pk = _packing(1000, 5)
    s = _system(pk, 256)
    try:
        print("autotune_fire", flush=True)
        got = s.autotune_fire(native.fire_params(ftol=1e-12), iterations=30)
        assert s.team_info() == (2, 0) and got["path"] == "list" and got["shape"] in (1, 2, 4, 8)
        s.gd_steps(5)
        assert s.team_info() == (3, 0)
        with pytest.raises(native.SpherocylsError):
            s.autotune_fire(native.fire_params(max_move=0.06), iterations=10)
        s.gd_steps(5)
        assert s.team_info() == (4, 0)
        s.set_small_fire(0)
        s.autotune_fire(native.fire_params(ftol=1e-12), iterations=30)
        s.gd_steps(5)
        assert s.team_info() == (4, 0)
    finally:
        s.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_packings_that_finished_before_another_gave_up(precision):
    """Of a batch only one packing runs out of room; the others finish in the
    team, the launches per step then pass them over, and the final evaluation,
    and the steps after it, are theirs too."""
    packs = [_packing(300, 4), _packing(1000, 1, discs=2, radius=3.0), _packing(100, 5),
             _packing(700, 6)]
    params = native.fire_params(dt0=0.05, dt_max=0.5, max_move=0.02, ftol=1e-12, max_iter=60)
    side = np.concatenate([np.full(p.n, p.L) for p in packs])
    for name in ("fire", "descent"):
        out = []
        for small in (256, 0):
            print("finished before,", name, precision, small, flush=True)
            s = _system(packs, small)
            try:
                s.set_precision(precision)
                s.set_dynamics(step=0.05)
                if name == "fire":
                    s.fire(params, check=False)
                else:
                    s.gd_steps(60)
                assert s.team_info() == ((1, native.SC_TEAM_NO_ROOM) if small else (0, 0))
                box = [s.box(k) for k in range(s.npack)]
                out.append((s.positions(), s.forces(), box))
                s.set_dynamics(strain_rate=1e-3, step=0.01)
                s.strain_steps(3)
                out.append((s.positions(), s.forces(), box))
            finally:
                s.close()
        tol = TOL if precision == "fp64" else 1e-5  # (FP32 pairs: 6e-8 of a force a step)
        for a, b in ((out[0], out[2]), (out[1], out[3])):
            _same(a, b, side, tol)
            for p, q in zip(a[2], b[2]):
                assert q["ncontacts"] > 50 and p["ncontacts"] == pytest.approx(q["ncontacts"], abs=2)
                assert p["E"] == pytest.approx(q["E"], rel=1e-3)


def test_packings_that_finished_before_a_resort():
    """Without graphs the launches per step re-sort the bank every 240
    iterations; packings that had finished (two of these jammed discs', whose
    descent has moved them far from their cells in the bank) keep their forces."""
    packs = []
    for n, phi, seed in ((60, 1.0, 1), (200, 1.1, 4), (400, 0.9, 6), (300, 0.88, 7)):
        R, A = configs.bidisperse(n, aspect=1.0)
        packs.append(configs.make_packing(R, A, phi, seed, f"N={n} phi {phi}"))
    params = native.fire_params(dt0=0.05, dt_max=0.5, max_move=0.02, ftol=1e-4, max_iter=2000)
    out = []
    for graphs in (False, True):
        print("re-sort", graphs, flush=True)
        s = _system(packs, 0)
        try:
            s.set_graphs(graphs)
            s.set_dynamics(step=0.1)
            s.gd_steps(500)
            it, _, _ = s.fire(params, check=False)
            out.append((it, s.positions(), s.forces(), [s.box(k) for k in range(4)]))
        finally:
            s.close()
    it = out[1][0]
    assert it[0] < 240 and it[1] < 240 and it[2] > 270 and it[3] > 270
    n = packs[0].n + packs[1].n  # (the re-sorted others' sums run in another order)
    np.testing.assert_array_equal(out[0][0][:2], it[:2])
    side = np.concatenate([np.full(p.n, p.L) for p in packs[:2]])
    _same(*[([v[:n] for v in o[1]], [v[:n] for v in o[2]]) for o in out], side, 1e-7)
    for p, q in zip(out[0][3][:2], out[1][3][:2]):
        assert q["ncontacts"] > 100 and p["ncontacts"] == q["ncontacts"]


@pytest.mark.parametrize("n,steps,every", [
    (100, 50, 20), (700, 50, 50), (700, 50, 7), (700, 4100, 1900), (4096, 60, 59)])
def test_the_box_keeps_the_last_record(n, steps, every):
    """Energy and stress of the box after sheared steps are those of the last
    recorded state (here of several launches, too)."""
    pk = _packing(n, 8, phi=0.84)
    out = []
    for small in (256, 0):
        print("last record", n, steps, every, small, flush=True)
        s = _system(pk, 0)
        try:
            s.fire(native.fire_params(dt0=0.05, dt_max=0.5, max_move=0.02, max_iter=200), check=False)
            s.set_small_fire(small)
            s.set_dynamics(strain_rate=1e-4, step=0.01)
            se = s.strain_steps(steps, every)
            assert s.team_steps() == (steps if small else 0)
            box = s.box(0)
            out.append([box[k] for k in native.SE_FIELDS])
            np.testing.assert_array_equal(out[-1], se[-1, 0])
        finally:
            s.close()
    np.testing.assert_allclose(out[0], out[1], rtol=0, atol=1e-7 * np.abs(out[1][:-1]).max())
