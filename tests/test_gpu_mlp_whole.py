"""Whole-network kernels against the launch-per-layer form (which per-class timing selects): the same sums
in the same order, so the same bits, at the edges of the 32-row and 32-column tiles."""
import numpy as np
import pytest

import mstcfd as M

pytestmark = pytest.mark.gpu


def run(per_layer, n_in, width, hidden, n_out, rows, n):
    rng = np.random.default_rng(n_in + width + rows)
    X = rng.uniform(-1, 1, (n, n_in)).astype(np.float32)
    T = rng.uniform(-1, 1, (n, n_out)).astype(np.float32)
    net = M.MLP(n_in, width, hidden, n_out, seed=5)
    f = lambda k, lo, hi: rng.uniform(lo, hi, k).astype(np.float32)
    net.set_scaling(f(n_in, -0.5, 0.5), f(n_in, 0.5, 2), f(n_out, -0.5, 0.5), f(n_out, 0.5, 2))
    net.set_data(X, T)
    net.timing(per_layer)
    out = [net.forward(X[:rows])]
    g, loss = net.gradient(X[:rows], T[:rows])
    loss2 = net.train(3, batch=rows, lr=1e-2)
    net.set_params(net.get_params() * np.float32(0.5))
    net.train(2, batch=rows, lr=1e-2)
    net.timing(not per_layer)  # and the other form goes on from there
    net.train(1, batch=rows, lr=1e-2)
    net.timing(per_layer)
    net.train(1, batch=rows, lr=1e-2)
    out += [g, np.array([loss, loss2]), net.get_params()]
    net.close()
    return out


@pytest.mark.parametrize("n_in,width,hidden,n_out,rows,n", [
    (4, 128, 4, 4, 1000, 3000), (1, 1, 1, 1, 1, 1), (3, 31, 2, 5, 31, 31), (9, 33, 1, 32, 33, 100), (64, 127, 2, 31, 65, 64),
    (7, 64, 3, 3, 512, 513), (4, 96, 5, 4, 20000, 20000), (8, 128, 16, 8, 257, 1000), (4, 129, 1, 4, 70, 70),
    (4, 40, 2, 33, 70, 70)])
def test_whole_network_kernels_match_per_layer_launches(n_in, width, hidden, n_out, rows, n):
    rows = min(rows, n)
    print(f"mlp {n_in}-{width}x{hidden}-{n_out}, {rows} of {n} rows", flush=True)
    a, b = (run(p, n_in, width, hidden, n_out, rows, n) for p in (False, True))
    for x, y in zip(a, b):
        assert np.all(np.isfinite(x)) and np.array_equal(x, y)
