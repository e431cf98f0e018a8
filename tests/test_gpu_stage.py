"""Copies between host arrays and the device through the pinned slots: sizes
around the plain copy's limit, the slot size and the ring's length, the 32 to
64 bit flags, and callers on several threads (one has the ring, the others copy
plainly).  Values come back as they went in."""
import threading

import numpy as np
import pytest

from main_amd import systems as S
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
