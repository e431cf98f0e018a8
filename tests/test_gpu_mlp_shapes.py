"""The surrogate's products at the edges of their tiles: sizes that are not
multiples of 16 or 32, one row, ragged batches, more layers than one gradient
launch takes, buffers reused after a larger batch; and sizes on both sides of
the 4,096 tiles of 16 x 16 from which a product takes tiles of 32 x 32.

Tolerance: the reference rounds the same operands to BF16 and sums in FP64; the
FP32 sums differ by about 1e-7, which moves about 1e-4 of the BF16 roundings of
the next layer by 2^-9 of a value, so about 4e-5 a product and 1e-3 through the
deepest network here; asserted at 2e-3.
"""
import numpy as np
import pytest

from main_amd.surrogate import Surrogate, gemm_bf16
from tests import mlp_reference as M

pytestmark = pytest.mark.gpu


def _problem(rows, n_in, n_out, seed):
    rng = np.random.default_rng(seed)
    x = rng.normal(size=(rows, n_in)).astype(np.float32)
    t = rng.normal(size=(rows, n_out)).astype(np.float32)
    return x, t, rng.uniform(0.5, 1.5, size=n_out).astype(np.float32)


@pytest.mark.parametrize("rows,n_in,hidden,layers,n_out", [
    (1, 1, 1, 1, 1), (1, 8, 64, 2, 33), (17, 5, 20, 1, 15), (31, 33, 100, 3, 65), (64, 8, 256, 3, 2049), (65, 8, 31, 9, 16)])
def test_gradients_at_tile_edges(rows, n_in, hidden, layers, n_out):
    net = Surrogate(n_in=n_in, n_hidden=hidden, n_layers=layers, n_out=n_out, seed=5)
    try:
        net.loss_grad_raw(*_problem(97, n_in, n_out, 3))   # the buffers of a larger batch, then reused
        x, t, w = _problem(rows, n_in, n_out, 4)
        loss, g = net.loss_grad_raw(x, t, w)
        f = lambda a: a.astype(np.float64)
        lr, gr = M.loss_grad(f(net.params()), net.dims(), f(x), f(t), f(w), bf16=True)
        assert abs(loss - lr) <= 2e-3 * lr
        assert np.linalg.norm(g - gr) <= 2e-3 * np.linalg.norm(gr)
        H, _ = M.forward(f(net.params()), net.dims(), f(x), bf16=True)
        assert np.max(np.abs(net.forward_raw(x) - H[-1])) <= 2e-3 * np.max(np.abs(H[-1]))
    finally:
        net.close()


@pytest.mark.parametrize("n,batch", [(1, 4), (33, 33), (50, 16), (70, 64)])
def test_an_epoch_is_adam_on_its_batches(n, batch):
    """Each step's parameters from the gradients the network reports for that
    step's rows, FP32 Adam in numpy: a few FP32 roundings of a step of size lr."""
    x, t, w = _problem(n, 8, 40, 6)
    seed, lr = 11, 1e-2
    net, twin = (Surrogate(n_in=8, n_hidden=48, n_layers=2, n_out=40, seed=9) for _ in range(2))
    try:
        losses = net.train_raw(x, t, w, batch=batch, epochs=2, lr=lr, seed=seed)
        p = twin.params().astype(np.float64)
        m, v, step, mask = np.zeros_like(p), np.zeros_like(p), 0, (1 << 64) - 1
        for ep in range(2):
            order, s = list(range(n)), ((seed + 1) * 6364136223846793005 + ep * 1442695040888963407) & mask
            for i in range(n - 1, 0, -1):
                s = (s * 6364136223846793005 + 1442695040888963407) & mask
                j = (s >> 33) % (i + 1)
                order[i], order[j] = order[j], order[i]
            total = 0.0
            for b in range(0, n, batch):
                q = order[b:b + batch]
                twin.set_params(p.astype(np.float32))
                loss, g = twin.loss_grad_raw(x[q], t[q], w)
                total += loss * len(q)
                step += 1
                m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g.astype(np.float64) ** 2
                p = (p - lr * (m / (1 - 0.9 ** step)) / (np.sqrt(v / (1 - 0.999 ** step)) + 1e-8)).astype(np.float32)
                p = p.astype(np.float64)
            assert abs(losses[ep] - total / n) <= 1e-3 * total / n
        # FP32 moments and bias corrections (1 - 0.999^t in FP32: 6e-5 relative at t = 1, halved by the root)
        d = np.abs(net.params() - p)
        assert np.median(d) <= 1e-4 * lr and np.quantile(d, 0.99) <= 1e-2 * lr
    finally:
        net.close()
        twin.close()


def _tiles(m, n):
    return (m + 31) // 32 * 2 * ((n + 15) // 16)


@pytest.mark.parametrize("m,n,k,wide", [(1000, 1008, 33, False), (1024, 1024, 32, True), (1037, 1045, 70, True),
                                        (2049, 513, 1, True), (4097, 241, 64, True), (33, 32700, 45, True)])
def test_products_of_wide_tiles(m, n, k, wide):
    """FP32 sums of exact products of BF16 values: their rounding, as the small products'."""
    assert (_tiles(m, n) >= 4096) == wide
    rng = np.random.default_rng(m + n + k)
    A, B = rng.normal(size=(m, k)).astype(np.float32), rng.normal(size=(k, n)).astype(np.float32)
    C, _ = gemm_bf16(A, B)
    a, b = M.to_bf16(A), M.to_bf16(B)
    assert np.max(np.abs(C - a @ b) / (np.abs(a) @ np.abs(b))) < 1e-6


@pytest.mark.parametrize("hidden,rows", [(256, (8192, 545, 1025, 480, 3)), (200, (4129, 5057, 512)), (31, (545, 97))])
def test_screening_of_many_rows(hidden, rows):
    """Batches one after the other on one network: wide tiles in some layers (480
    rows: none; 545: the output layer; 5,057 and more: the hidden ones of 200
    or 256 units too), buffers kept from a larger batch, ragged edges."""
    net = Surrogate(n_in=8, n_hidden=hidden, n_layers=2, n_out=2049, seed=8)
    try:
        flat = net.params().astype(np.float64)
        for n in rows:
            x = np.random.default_rng(n).normal(size=(n, 8)).astype(np.float32)
            H, _ = M.forward(flat, net.dims(), x.astype(np.float64), bf16=True)
            assert np.max(np.abs(net.forward_raw(x) - H[-1])) <= 2e-3 * np.max(np.abs(H[-1])), n
    finally:
        net.close()
