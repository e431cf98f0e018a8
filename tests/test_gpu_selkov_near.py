"""The Selkov near engine's forms against each other: particles that matter in
registers (the default, also with a large guard), the spheres leaving the
margin of their start in mid-launch (a small guard: the general form takes over
at that step), and more particles than the registers hold (large spheres and a
guard that puts the first launch's count, made here as the engine makes it, at
the registers' 2,048, one beyond, and far beyond: the general form throughout).

The guard only sets which particles count as near, so the trajectories agree to
the rounding of the sphere sums, whose order follows the near set: about 1e-16
of a sum a step, and less than a factor 1e3 of growth over these 80 steps;
asserted at 1e-11 (positions), 1e-10 (velocities).  Species are equal.
"""
import numpy as np
import pytest

from main_amd import systems as S
from main_amd.selkov import SelkovEngine

pytestmark = pytest.mark.gpu


def _run(guard, sort_step, rates):
    p = S.selkov_params(L=24.0, rho=10.0, NG=24 ** 3, T=2.0, RPfg=rates[0], RPgf=rates[1])
    s = S.selkov_initial_state(p, seed=12)
    s["dm"][:, 3] = 0.1   # the dimer drifts 0.01 an interval
    e = SelkovEngine(p, rng_mode=1, seed=5, sort_step=sort_step, sphere_guard=guard)
    try:
        e.set_state(s)
        e.run(4)
        return e.get_state()
    finally:
        e.close()


@pytest.mark.parametrize("rates", [(1.0, 0.0), (0.6, 0.3)])
@pytest.mark.parametrize("sort_step", [10000, 40])
def test_near_engine_forms_agree(sort_step, rates):
    ref = _run(1.0, sort_step, rates)
    for guard in (0.05, 3.2):
        g = _run(guard, sort_step, rates)
        assert np.array_equal(g["flag"], ref["flag"]), guard
        for k, tol in (("x", 1e-11), ("y", 1e-11), ("z", 1e-11), ("vx", 1e-10), ("vy", 1e-10), ("vz", 1e-10)):
            assert np.max(np.abs(g[k] - ref[k])) <= tol, (guard, k)
        assert np.max(np.abs(g["dm"][:, :6] - ref["dm"][:, :6])) <= 1e-11, guard


HELD = 2048   # entries of the register form


def _large_spheres():
    p = S.selkov_params(L=24.0, rho=10.0, NG=24 ** 3, T=10.0, RPfg=0.6, RPgf=0.3, Rc=3.0, Rn=5.0, Dcn=10.0)
    s = S.selkov_initial_state(p, seed=12)
    s["dm"][:, 3] = 0.02
    # how far a particle stays from a cutoff if it flies straight at it for a launch
    v = np.sqrt(s["vx"] ** 2 + s["vy"] ** 2 + s["vz"] ** 2) * p["MDt"] * p["MPCtstep"]
    gap = np.full(p["NT"], np.inf)
    for i, R in enumerate((p["Rc"], p["Rn"])):
        d = [s[k] - s["dm"][i, j] for j, k in enumerate("xyz")]
        r = np.sqrt(sum((a - b * np.rint(a / b)) ** 2 for a, b in zip(d, p["box"])))
        gap = np.minimum(gap, r - R * p["cutoff"] - v)
    return p, s, np.sort(gap)


def _run_large(p, s, guard, sort_step):
    e = SelkovEngine(p, rng_mode=1, seed=5, sort_step=sort_step, sphere_guard=guard)
    try:
        e.set_state(s)
        e.run(2)
        return e.get_state()
    finally:
        e.close()


@pytest.mark.parametrize("sort_step", [10000, 20])
def test_more_particles_than_the_registers_hold(sort_step):
    """A launch keeps the particles within 0.1 guard of a cutoff after its flight."""
    p, s, gap = _large_spheres()
    guards = [0.5] + [10.0 * 0.5 * (gap[n - 1] + gap[n]) for n in (HELD, HELD + 1)] + [2.0]
    counts = [int(np.sum(gap <= 0.1 * g)) for g in guards]
    assert counts[0] < HELD - 300 and counts[1:3] == [HELD, HELD + 1] and counts[3] > HELD + 500
    ref = _run_large(p, s, guards[0], sort_step)
    for g in guards[1:]:
        o = _run_large(p, s, g, sort_step)
        assert np.array_equal(o["flag"], ref["flag"]), g
        for k, tol in (("x", 1e-11), ("y", 1e-11), ("z", 1e-11), ("vx", 1e-10), ("vy", 1e-10), ("vz", 1e-10)):
            assert np.max(np.abs(o[k] - ref[k])) <= tol, (g, k)
        assert np.max(np.abs(o["dm"][:, :6] - ref["dm"][:, :6])) <= 1e-11, g


def test_near_engine_starts_before_the_far_stream():
    """The near engine needs a CU to itself: started after the far particles'
    2,048 workgroups it waits for their first round, and the second stream gains
    nothing (0.495 ms an interval at this size, 0.508 in one stream); started
    first, 0.384 ms."""
    p = S.selkov_params(L=50.0, rho=10.0, NG=int(0.8 * 50 ** 3))
    e = SelkovEngine(p, rng_mode=1, seed=3)
    try:
        e.set_state(S.selkov_initial_state(p, seed=3), cstep=0)
        ms = {True: [], False: []}
        for _ in range(4):
            for on in (False, True):
                e.set_overlap(on)
                e.run(32)
                ms[on].append(e.kernel_ms()["run_ms"])
    finally:
        e.close()
    assert min(ms[True]) < 0.88 * min(ms[False]), ms
