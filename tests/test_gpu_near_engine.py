"""Edges of the near engines against the oracle: inside entries beyond the ones
LDS holds (one dimer and two), entries in more than two neighbour lists with
every step in the general form's reach, and the far particles' sphere culling
at its threshold and beyond one wave's worth of spheres.

Compared as tests/parity_cases.py states: integers and lists equal, positions
and velocities within 1e-12 of max(|reference|, scale); the sums over a list
are the only reordered arithmetic (some 1e-15 of a sum a step, tens of steps).
"""
import numpy as np
import pytest

from main_amd.tour import cell_tour
from tests.parity_cases import collective_parity_case, small_collective_params

pytestmark = pytest.mark.gpu

LDS_ENTRIES = 2304
BIG = dict(rhoa=16.0, Rc=2.0, Rn=4.0, Dcn=6.5)

CASES = {
    "one_dimer_beyond_lds": dict(p=dict(Lx=20.0, Ly=18.0, Lz=22.0, **{**BIG, "rhoa": 28.0}), inside=LDS_ENTRIES + 1),
    "two_dimers_beyond_lds": dict(p=dict(numdims=2, Lx=26.0, Ly=26.0, Lz=20.0, **BIG), inside=LDS_ENTRIES + 1),
    "three_dimers_shared_lists": dict(p=dict(numdims=3, Lx=14.0, Ly=14.0, Lz=14.0, rhoa=8.0, skinrad=1.0, EbN=0.1),
                                      near_mode=0, shared=3),
    "seven_dimers_not_culled": dict(p=dict(numdims=7, Lx=28.0, Ly=28.0, Lz=14.0, rhoa=4.0)),
    "forty_dimers_culled": dict(p=dict(numdims=40, Lx=53.0, Ly=50.0, Lz=18.0, rhoa=4.0, sort_step=10)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_near_engine_edges_match_oracle(name):
    c = CASES[name]
    p = small_collective_params(**c["p"])
    r = collective_parity_case(ncoll=2, seed=31, p=p, flags_mix=True, near_mode=c.get("near_mode"),
                               tour=cell_tour(*(int(v) for v in p["box"])))
    lists = r["lists"]
    assert len(lists["in_list"]) >= c.get("inside", 0)
    members = np.concatenate([lists["nb"][k, i, :lists["nbnum"][k, i]] for k in range(p["numdims"]) for i in range(2)])
    assert np.max(np.unique(members, return_counts=True)[1]) >= c.get("shared", 1)
    assert r["ok"], f"{name}: {r['summary']}"
