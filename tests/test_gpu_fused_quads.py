"""The fused kernel on FP64 quadrilaterals either side of the size where its blocks get twice the lanes (256 blocks): the
face strategy's bits, and at 468 blocks, where the wide blocks leave one patch per compute unit and had made it 13 %
slower than the patch kernels, a step no longer than theirs."""
import time

import numpy as np
import pytest

import mstcfd as M
from helpers import cons, quad_grid

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,prec", [(256, M.PREC_FP64), (257, M.PREC_FP64), (346, M.PREC_FP64), (346, M.PREC_MIXED),
                                    (362, M.PREC_MIXED), (363, M.PREC_MIXED)])
def test_fused_quadrilaterals(n, prec):
    m = M.Mesh.from_raw(quad_grid(n, bc=M.BC_WALL, h=0.05, jitter=0.2, seed=4))
    print(f"fused quadrilaterals: {m.n_cells} cells, precision {prec}", flush=True)
    rng = np.random.default_rng(1)
    k = m.n_cells
    Q = cons(rng.uniform(0.95, 1.05, k), rng.uniform(-0.1, 0.1, (k, 2)), rng.uniform(0.95, 1.05, k))
    s = M.Solver(m, M.make_config(order=2, scheme=M.ROE, limiter=M.LIM_MINMOD, rk=2, cfl=1e-3, precision=prec,
                                  q_inlet=list(Q[0])))
    got, t = {}, {}
    for st in (M.STRATEGY_FACE, M.STRATEGY_PATCH, M.STRATEGY_FUSED):
        s.strategy = st
        s.set_state(Q)
        s.step(3)
        got[st] = s.get_state(), s.residual_norms()
        s.step(5)
        t[st] = np.inf
        for _ in range(10):
            t0 = time.perf_counter()
            s.step(20)
            t[st] = min(t[st], 1e6 * (time.perf_counter() - t0) / 20)
    s.close()
    for st in got:
        assert all(np.array_equal(a, b) for a, b in zip(got[st], got[M.STRATEGY_FACE]))
    print({st: round(v, 2) for st, v in t.items()}, flush=True)
    if n == 346:
        assert t[M.STRATEGY_FUSED] <= 1.05 * t[M.STRATEGY_PATCH]
