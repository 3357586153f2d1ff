"""One batch stepped with every strategy in turn (queues and one item per block, in every order) equals single contexts
bit for bit: uneven cases, Roe and AUSM, one of them frozen on the way."""
import itertools

import numpy as np
import pytest

import mstcfd as M
from helpers import cons

pytestmark = pytest.mark.gpu

ALL = (M.STRATEGY_FACE, M.STRATEGY_CELL, M.STRATEGY_PATCH, M.STRATEGY_FUSED)


@pytest.mark.parametrize("prec", [M.PREC_FP64, M.PREC_MIXED])
@pytest.mark.parametrize("order", [1, 2])
def test_strategies_in_turn(order, prec):
    bc = (M.BC_INLET, M.BC_OUTLET, M.BC_WALL, M.BC_SYMMETRY)
    meshes = [M.Mesh.gen_tri(nx, ny, 0, 2, 0, 1, 0.1, nx, bc) for nx, ny in ((1, 1), (40, 31), (13, 10), (70, 50))]
    lim = M.LIM_MINMOD if order == 2 else M.LIM_NONE
    rng = np.random.default_rng(order)
    states = [cons(rng.uniform(0.95, 1.05, m.n_cells), rng.uniform(-0.1, 0.1, (m.n_cells, 2)),
                   rng.uniform(0.95, 1.05, m.n_cells)) for m in meshes]
    cfgs = [M.make_config(scheme=(M.ROE, M.AUSM)[i % 2], order=order, limiter=lim, rk=2, cfl=0.3, precision=prec,
                          q_inlet=list(states[0][0])) for i in range(4)]
    seq = [s for a, b in itertools.permutations(ALL, 2) for s in (a, b)]
    b = M.Batch(meshes, cfgs)
    for i, q in enumerate(states):
        b.set_state(i, q)
    for k, st in enumerate(seq):
        if k == 6:
            b.set_active(np.array([1, 1, 0, 1], np.uint8))
        if k == 9:
            b.set_active(np.ones(4, np.uint8))
        b.strategy = st
        b.step(1)
    print(f"batch strategies in turn: order {order}, precision {prec}, {len(seq)} steps", flush=True)
    for i in range(4):
        s = M.Solver(meshes[i], cfgs[i])
        s.set_state(states[i])
        for k in range(len(seq)):
            if not (i == 2 and 6 <= k < 9):
                s.step(1)
        assert np.all(np.isfinite(s.get_state()))
        assert np.array_equal(b.get_state(i), s.get_state()), i
        s.close()
    b.close()
