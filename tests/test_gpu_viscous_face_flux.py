"""The face fluxes a viscous context holds are those of its last stage, whichever route the stage took: face_flux_values
and residual_update after solve, steps, a new state, another configuration and a warm start give what the face strategy
gives, bit for bit."""
import numpy as np
import pytest

import mstcfd as M
from helpers import cons, quad_grid

pytestmark = pytest.mark.gpu

MESHES = {
    "tri": lambda: M.Mesh.gen_tri(31, 20, 0, 3, 0, 2, 0.15, 7, (M.BC_INLET, M.BC_OUTLET, M.BC_WALL, M.BC_SYMMETRY)),
    "periodic": lambda: M.Mesh.gen_tri(24, 24, -1, 1, -1, 1, 0.15, 3, (M.BC_PERIODIC,) * 4),
    "quad": lambda: M.Mesh.from_raw(quad_grid(20, bc=M.BC_WALL, h=0.05, jitter=0.2, seed=4)),
    "tet": lambda: M.Mesh.gen_tet(6, 5, 4, (0, 0, 0), (1, 0.8, 0.7), 0.15, 11,
                                  (M.BC_INLET, M.BC_OUTLET, M.BC_SYMMETRY, M.BC_WALL, M.BC_SYMMETRY, M.BC_WALL)),
}


def sequence(m, states, strategy, order, prec):
    cfg = lambda mu, p=prec: M.make_config(dim=m.dim, scheme=M.ROE, order=order, limiter=M.LIM_VANLEER, rk=3, precision=p,
                                           mu=mu, kappa=0.05 * (mu > 0), cv=2.5, q_inlet=list(states[0][0]))
    s = M.Solver(m, cfg(0.03))
    s.strategy = strategy
    s.set_state(states[0])
    s.set_dt(1e-4)
    out = []
    G = lambda: out.append(s.face_flux_values())
    s.solve()
    G()
    s.solve()
    s.residual_update()  # the fluxes of the solve before it
    out.append(s.get_new_state())
    s.update_new_to_old()
    G()
    s.step(2)
    G()
    s.set_state(states[1])  # (another buffer than the last stage's)
    G()
    s.solve()
    s.set_state(states[2])  # over the state that the fluxes are of
    G()
    s.solve()
    s.set_config(cfg(0.06))
    G()
    s.step(1)
    s.set_config(cfg(0.0, M.PREC_FP64))
    G()
    s.set_config(cfg(0.03))
    s.step(1)
    net = M.MLP(m.dim + 1, 16, 1, m.nv, seed=1)
    s.warm_start(net, [0.5])
    G()
    s.set_state(states[0])
    s.step(1)
    s.lusgs_step(1)
    G()
    net.close()
    s.close()
    return out


@pytest.mark.parametrize("order,prec", [(1, M.PREC_FP64), (2, M.PREC_FP64), (1, M.PREC_MIXED), (2, M.PREC_MIXED)])
@pytest.mark.parametrize("name", sorted(MESHES))
def test_face_fluxes_are_the_last_stages(name, order, prec):
    m = MESHES[name]()
    print(f"viscous face fluxes {name}: {m.n_cells} cells, order {order}, precision {prec}", flush=True)
    rng = np.random.default_rng(3)
    n = m.n_cells
    states = [cons(rng.uniform(0.95, 1.05, n), rng.uniform(-0.1, 0.1, (n, m.dim)), rng.uniform(0.95, 1.05, n)) for _ in range(3)]
    want = sequence(m, states, M.STRATEGY_FACE, order, prec)
    for st in (M.STRATEGY_PATCH, M.STRATEGY_AUTO):
        got = sequence(m, states, st, order, prec)
        for k, (g, w) in enumerate(zip(got, want)):
            assert np.all(np.isfinite(w)) and np.array_equal(g, w), (st, k)
