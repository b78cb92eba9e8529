"""Batches of packings that are a single member of a team each: they wait for
nobody, so any number runs in one launch (up to 128 particles with any mode,
FIRE of up to 256 where their teams of several would not fit the GPU), behind
larger packings' teams, and beside the launches of other threads.  Against the
launches per step; both sides evaluate the same formulas and differ in the order
of sums (a few units in the last place per step, below 1e-13 over 40 iterations,
with a factor of 1e4 left for contacts that amplify it)."""
import threading

import numpy as np
import pytest

from spherocyls_amd import configs, native

pytestmark = pytest.mark.gpu
TOL = 1e-9
PARAMS = dict(dt0=0.05, dt_max=0.5, max_move=0.02, ftol=1e-12, max_iter=40)


def _packs(sizes):
    made = {}
    for n in sizes:
        if n not in made:
            R, A = configs.bidisperse(n, aspect=1.5)
            made[n] = configs.make_packing(R, A, 0.84 if n > 9 else 0.2, 11 + n, f"N={n}")
    return [made[n] for n in sizes]


def _run(packs, small, calls):
    s = native.System(packs, pads=0.1)
    try:
        s.set_contact_model("two_point")
        s.set_small_fire(small)
        out = []
        for name in calls:
            if name == "fire":
                s.fire(native.fire_params(**PARAMS), check=False)
            else:
                s.gd_steps(40)
            out.append((s.positions(), s.forces()))
        return out, s.team_info()
    finally:
        s.close()


def _compare(a, b, packs):
    L = np.concatenate([np.full(p.n, p.L) for p in packs])
    for (pa, fa), (pb, fb) in zip(a, b):
        for u, v, side in zip(pa, pb, (L, L, 2 * np.pi)):
            d = u - v
            assert np.max(np.abs(d - side * np.round(d / side))) < TOL
        for u, v in zip(fa, fb):
            assert np.max(np.abs(u - v)) < TOL * max(1.0, np.max(np.abs(v)))


@pytest.mark.parametrize("sizes,calls,launches", [
    ((100,) * 700, ("fire", "descent"), 2),      # more than are resident at once
    ((1, 2, 64, 65, 128) * 150, ("fire", "descent"), 2),
    ((256, 129, 255, 193) * 80, ("fire",), 1),   # one member each
    ((128, 200, 256, 3) * 100, ("fire",), 1),
    ((700,) + (100,) * 600 + (65, 1500), ("fire", "descent"), 2),
    ((129, 64) * 250, ("descent",), 1)])
def test_batches_in_one_launch(sizes, calls, launches):
    packs = _packs(sizes)
    print("batch of", len(sizes), sorted(set(sizes)), flush=True)
    a, info = _run(packs, 256, calls)
    assert info == (launches, 0)
    b, info = _run(packs, 0, calls)
    assert info == (0, 0)
    _compare(a, b, packs)


def test_threads_beside_each_other():
    """Systems of single members and of teams of several on four threads give
    what each gives alone, bit for bit."""
    work = [_packs(s) for s in ((100,) * 40, (900,), (60, 128), (200, 70))]
    alone = [_run(p, 256, ("fire", "descent")) for p in work]
    got = [None] * len(work)

    def go(i):
        for _ in range(3):
            got[i] = _run(work[i], 256, ("fire", "descent"))

    threads = [threading.Thread(target=go, args=(i,)) for i in range(len(work))]
    print("threads", flush=True)
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, b in zip(alone, got):
        assert a[1] == b[1]
        for (pa, fa), (pb, fb) in zip(a[0], b[0]):
            for u, v in zip((*pa, *fa), (*pb, *fb)):
                np.testing.assert_array_equal(u, v)


def test_limit_on_the_size():
    """Below 256 the limit is a number of particles of every packing still
    advanced; at 256 there is none."""
    for sizes, limit, launches in (((100,), 99, 0), ((100,), 100, 1), ((60, 100), 64, 0),
                                   ((60, 64), 64, 1), ((700,), 255, 0), ((700,), 256, 1)):
        for call in ("fire", "descent"):
            print("limit", sizes, limit, call, flush=True)
            _, info = _run(_packs(sizes), limit, (call,))
            assert info == (launches, 0)
    s = native.System(_packs((300,)), pads=0.1)
    try:
        s.set_dynamics(strain_rate=1e-3, step=0.005)
        for limit, launches in ((200, 0), (255, 0), (256, 1)):
            s.set_small_fire(limit)
            s.strain_steps(50)
            assert s.team_info()[0] == launches
    finally:
        s.close()
