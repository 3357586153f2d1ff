"""Training as a replayed graph, on networks that take that route (width above 128, or more than 32 outputs; the smaller ones
run the whole-network kernels, kept here as a third case): replays against direct launches of the same calls bit for
bit, through what replaces the captured buffers, and against the CPU reference with test_gpu_mlp's bounds."""
import numpy as np
import pytest

import mlp_ref as R
import mstcfd as M

pytestmark = pytest.mark.gpu

NETS = [(160, 2, 4), (64, 2, 33), (128, 4, 4)]  # width, hidden layers, outputs


def make(width, hidden, n_out, seed):
    net = M.MLP(4, width, hidden, n_out, seed=seed)
    rng = np.random.default_rng(seed)
    f = lambda k, lo, hi: rng.uniform(lo, hi, k).astype(np.float32)
    sc = f(4, -0.5, 0.5), f(4, 0.5, 2), f(n_out, -0.5, 0.5), f(n_out, 0.5, 2)
    net.set_scaling(*sc)
    return net, sc


def data(n, n_out, seed):
    rng = np.random.default_rng(seed)
    X = rng.uniform(-1, 1, (n, 4)).astype(np.float32)
    k = np.arange(n_out)
    T = np.sin(X[:, :1] * (1 + k % 5) + X[:, 1:2]) * X[:, 2:3] + np.cos(k) * X[:, 3:]
    return X, T.astype(np.float32)


@pytest.mark.parametrize("width,hidden,n_out", NETS)
def test_full_batch_adam_replayed(width, hidden, n_out):
    X, T = data(500, n_out, 5)
    out = []
    for graph in (False, True):
        net, sc = make(width, hidden, n_out, 6)
        p0 = net.get_params().astype(np.float64)
        net.set_data(X, T)
        net.train(5, batch=500, lr=1e-3, graph=graph)
        out.append(net.get_params())
        layers = net.layers()
        net.close()
    assert np.array_equal(out[0], out[1])
    scd = [a.astype(np.float64) for a in sc]
    p, m, v = p0, np.zeros_like(p0), np.zeros_like(p0)
    for t in range(1, 6):
        _, g = R.loss_and_grad(p, layers, X.astype(np.float64), T.astype(np.float64), scd)
        p, m, v = R.adam(p, g, m, v, t, lr=1e-3)
    rel = np.linalg.norm((out[0] - p0) - (p - p0)) / np.linalg.norm(p - p0)
    print(f"4-{width}x{hidden}-{n_out}: 5 Adam steps, displacement rel. error {rel:.2e}", flush=True)
    assert rel <= 2e-3


@pytest.mark.parametrize("width,hidden,n_out", NETS)
def test_replay_survives_replaced_buffers(width, hidden, n_out):
    X1, T1 = data(6000, n_out, 7)
    X2, T2 = data(9000, n_out, 8)
    out = []
    for graph in (False, True):
        net, _ = make(width, hidden, n_out, 9)
        net.set_data(X1, T1)
        got = []
        for _ in range(3):
            got.append(net.train(4, batch=4096, lr=1e-3, graph=graph))
            net.forward(X2)  # uses the work buffers between replays
        net.gradient(*data(40000, n_out, 11))  # grows the work and the split buffers
        for _ in range(2):
            got.append(net.train(4, batch=4096, lr=1e-3, graph=graph))
        net.forward(data(200000, n_out, 10)[0])  # grows the work buffers again
        got.append(net.train(4, batch=4096, lr=1e-3, graph=graph))
        net.set_data(X2, T2)
        got.append(net.train(4, batch=4096, lr=1e-3, graph=graph))
        got.append(net.train(4, batch=1000, lr=1e-3, graph=graph))  # another batch
        got.append(net.train(4, batch=1000, lr=1e-2, graph=graph))  # another rate
        net.set_params(net.get_params() * np.float32(0.5))
        net.reset_optimizer()
        got.append(net.train(4, batch=1000, lr=1e-2, graph=graph))
        out.append((net.get_params(), np.array(got)))
        net.close()
    assert np.all(np.isfinite(out[0][0])) and np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("width,hidden,n_out", NETS)
def test_timed_steps_between_replays(width, hidden, n_out):
    X, T = data(20000, n_out, 12)
    out = []
    for timed in (False, True):
        net, _ = make(width, hidden, n_out, 13)
        net.set_data(X, T)
        for part in range(3):  # the middle part is launched directly when it is timed
            net.timing(timed and part == 1)
            net.train(3, batch=2048, lr=1e-3, graph=True)
        out.append(net.get_params())
        if timed:
            assert net.timing_get(M.MLP_K_GEMM_FWD)[0] == 3 * len(net.layers())
        net.close()
    assert np.array_equal(out[0], out[1])
