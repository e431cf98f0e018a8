"""Copies between host arrays and the device through the pinned slots: sizes
around the plain copy's limit, the slot size and the ring's length, the 32 to
64 bit flags, and callers on several threads (one has the ring, the others copy
plainly).  Values come back as they went in.  The parameters and the Selkov
state come out through the slots; the collective state goes in through them
too, so those round trips are of both directions."""
import threading

import numpy as np
import pytest

from main_amd import systems as S
from main_amd.collective import CollectiveEngine
from main_amd.selkov import SelkovEngine
from main_amd.surrogate import Surrogate

pytestmark = pytest.mark.gpu

SLOT = (2 << 20) // 4          # floats of a slot
LIMIT = (1 << 20) // 4         # below: the plain copy


def _net(nparam):
    """1 -> 1 -> n network: 2n + 2 parameters."""
    return Surrogate(n_in=1, n_hidden=1, n_layers=1, n_out=nparam // 2 - 1, seed=1)


def _round_trip(nparam, seed):
    net = _net(nparam)
    try:
        a = np.random.default_rng(seed).standard_normal(net.nparam).astype(np.float32)
        net.set_params(a)
        return np.array_equal(net.params(), a) and np.array_equal(net.params(), a)
    finally:
        net.close()


@pytest.mark.parametrize("nparam", [4, LIMIT - 2, LIMIT, SLOT, SLOT + 2, 2 * SLOT - 2, 4 * SLOT + 6, 16 * SLOT + 2,
                                    17 * SLOT, 33 * SLOT + 10])
def test_parameters_round_trip(nparam):
    assert _round_trip(nparam, nparam)


@pytest.mark.parametrize("L", [16, 31, 44])
def test_selkov_state_round_trip(L):
    p = S.selkov_params(L=float(L), rho=10.0, NG=L ** 3)
    s = S.selkov_initial_state(p, seed=L)
    s["flag"] = np.random.default_rng(L).permutation(s["flag"])
    e = SelkovEngine(p, rng_mode=1, seed=3)
    try:
        e.set_state(s)
        g = e.get_state()
        for k in ("x", "y", "z", "vx", "vy", "vz", "fx", "flag"):
            assert np.array_equal(g[k], s[k]), k
    finally:
        e.close()


def test_copies_on_several_threads():
    ok = [None] * 4

    def work(i):
        ok[i] = all(_round_trip(6 * SLOT + 2 * i, 10 * i + r) for r in range(3))

    th = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert ok == [True] * 4


def _collective_round_trip(L, rounds=1):
    """Six FP64 arrays and the flags in and out, fresh values each round."""
    p = S.collective_params(Lx=float(L), Ly=float(L), Lz=float(L), numdims=1, rhoa=10.0)
    e = CollectiveEngine(p, rng_mode=1, seed=3)
    rng = np.random.default_rng(L)
    s = {**S.collective_dimers(p, seed=L), "cstep": 0}
    ok = True
    try:
        for _ in range(rounds):
            s.update({k: L * rng.random(p["NT"]) for k in ("x", "y", "z", "vx", "vy", "vz")})
            s["flag"] = rng.integers(0, 3, p["NT"]).astype(np.int32)
            e.set_state(s)
            g = e.get_state()
            ok = ok and all(np.array_equal(g[k], s[k]) for k in ("x", "y", "z", "vx", "vy", "vz", "flag"))
    finally:
        e.close()
    return ok


@pytest.mark.parametrize("L", [13, 14, 28, 45, 61])   # 0.99 and 1.2 (the limit between), 11, 47 and 118 MB: up to four times round the ring
def test_collective_state_round_trip(L):
    assert _collective_round_trip(L, 2)


def test_uploads_on_several_threads():
    ok = [None] * 3

    def work(i):
        ok[i] = _collective_round_trip(40 + i, 3)

    th = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert ok == [True] * 3
