"""A context's patches follow its configuration: small meshes switched between FP64 and the mixed form have the patches of
a context created so (counted by the bytes of a patch launch), and every strategy still gives the same bits."""
import numpy as np
import pytest

import mstcfd as M
from helpers import cons

pytestmark = pytest.mark.gpu

MIX2 = (M.BC_INLET, M.BC_OUTLET, M.BC_WALL, M.BC_SYMMETRY)
MESHES = {
    "162 3D": lambda: M.Mesh.gen_tet(3, 3, 3, (0, 0, 0), (1, 1, 1), 0.1, 3, MIX2 + (M.BC_WALL,) * 2),
    "13182 3D": lambda: M.Mesh.gen_tet(13, 13, 13, (0, 0, 0), (1, 1, 1), 0.1, 3, MIX2 + (M.BC_WALL,) * 2),
    "322": lambda: M.Mesh.gen_tri(23, 7, 0, 4, 0, 2, 0.1, 7, MIX2),
}


@pytest.mark.parametrize("order,mu", [(1, 0.0), (2, 0.0), (2, 0.01)])
@pytest.mark.parametrize("name", sorted(MESHES))
def test_patches_follow_the_configuration(name, order, mu):
    m = MESHES[name]()
    rng = np.random.default_rng(8)
    n = m.n_cells
    print(f"patches of a changed configuration {name}: {n} cells, order {order}, mu {mu}", flush=True)
    Q = cons(rng.uniform(0.95, 1.05, n), rng.uniform(-0.1, 0.1, (n, m.dim)), rng.uniform(0.95, 1.05, n))
    cfg = lambda prec: M.make_config(dim=m.dim, scheme=M.AUSM, order=order, limiter=M.LIM_MINMOD if order == 2 else M.LIM_NONE,
                                     rk=2, cfl=0.2, precision=prec, q_inlet=list(Q[0]), mu=mu, kappa=mu, cv=2.5)

    def run(s, st):
        s.strategy = st
        s.set_state(Q)
        s.step(1)
        r = s.residual_norms()
        s.step(3)
        return s.get_state(), r, s.residual_norms(), np.array(s.compute_dt(0.2)), np.array(s.algorithmic_bytes(M.K_PATCH))

    both = (M.PREC_FP64, M.PREC_MIXED)
    want = {}
    for prec in both:
        s = M.Solver(m, cfg(prec))
        want[prec] = run(s, M.STRATEGY_FACE)
        s.close()
    for first in both:
        s = M.Solver(m, cfg(first))
        for prec in (first, both[first == both[0]], first):
            s.set_config(cfg(prec))
            for st in (M.STRATEGY_PATCH, M.STRATEGY_FUSED, M.STRATEGY_FACE):
                got = run(s, st)
                assert all(np.array_equal(g, w) for g, w in zip(got, want[prec])), (first, prec, st)
        if mu == 0 and order == 1:
            s.set_config(cfg(M.PREC_FP64))  # the implicit driver's residual reads the same tables
            s.set_state(Q)
            s.set_steady_driver(M.STEADY_LUSGS, 0.5, 1.0)
            s.lusgs_step(2)
            t = M.Solver(m, cfg(M.PREC_FP64))
            t.set_state(Q)
            t.set_steady_driver(M.STEADY_LUSGS, 0.5, 1.0)
            t.lusgs_step(2)
            assert np.array_equal(s.get_state(), t.get_state()) and np.array_equal(s.residual_norms(), t.residual_norms())
            t.close()
        s.close()
