"""The surrogate's training buffers: laid out for the call's own batch whatever
an earlier call was, bounded whatever the epoch's length, and an epoch that is
taken in parts is the same epoch.

One row a batch, so a twin trained row by row in the epoch's order makes the
same products in the same order: parameters and losses are equal bit for bit.
"""
import ctypes as C

import numpy as np
import pytest

from main_amd.surrogate import Surrogate
from tests.test_zz_no_alloc import _hip

pytestmark = pytest.mark.gpu


def _free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert _hip().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _problem(rows, n_in, n_out):
    rng = np.random.default_rng(rows + n_in)
    x = rng.normal(size=(rows, n_in)).astype(np.float32)
    t = rng.normal(size=(rows, n_out)).astype(np.float32)
    return x, t, np.full(n_out, 1.0 / n_out, np.float32)


def _order(n, seed):
    """Rows of a run's first epoch: shuffled by a 64-bit linear congruential generator."""
    order, mask = list(range(n)), (1 << 64) - 1
    s = (seed + 1) * 6364136223846793005 & mask
    for i in range(n - 1, 0, -1):
        s = (s * 6364136223846793005 + 1442695040888963407) & mask
        j = (s >> 33) % (i + 1)
        order[i], order[j] = order[j], order[i]
    return order


def test_small_batches_after_a_large_one():
    """A gradient of 4,096 rows, then epochs of small batches over them."""
    x, t, w = _problem(4096, 8, 33)
    net, fresh = (Surrogate(n_in=8, n_hidden=32, n_layers=2, n_out=33, seed=4) for _ in range(2))
    try:
        net.loss_grad_raw(x, t, w)
        for batch in (1, 50):
            before = _free_bytes()
            losses = net.train_raw(x, t, w, batch=batch, epochs=1, lr=1e-3, seed=2)
            # the input rows, both layouts, 128 bytes each of 32 a batch; shares and losses; 2 MB pages
            assert before - _free_bytes() <= 4096 * 32 * 128 + (16 << 20)
            assert np.array_equal(losses, fresh.train_raw(x, t, w, batch=batch, epochs=1, lr=1e-3, seed=2))
            assert np.array_equal(net.params(), fresh.params())
    finally:
        net.close()
        fresh.close()


@pytest.mark.parametrize("n,n_in", [(26, 20000), (27, 20000), (60, 20000), (30, 8)])
def test_an_epoch_in_parts(n, n_in):
    """26 steps of 20,000 inputs are held at once: the epoch in one part, one
    step over, three parts, and one part of few inputs."""
    x, t, w = _problem(n, n_in, 17)
    net, twin = (Surrogate(n_in=n_in, n_hidden=16, n_layers=1, n_out=17, seed=6) for _ in range(2))
    try:
        losses = net.train_raw(x, t, w, batch=1, epochs=1, lr=1e-3, seed=3)
        total = 0.0
        for q in _order(n, 3):
            total += twin.train_raw(x[q:q + 1], t[q:q + 1], w, batch=1, epochs=1, lr=1e-3, seed=3)[0]
        assert losses[0] == total / n
        assert np.array_equal(net.params(), twin.params())
    finally:
        net.close()
        twin.close()
