"""The Selkov near engine's forms against each other: particles that matter in
registers (the default), the spheres leaving the margin of their start in
mid-launch (a small guard: the general form takes over at that step), and more
particles than the registers hold (a large guard: the general form throughout).

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
