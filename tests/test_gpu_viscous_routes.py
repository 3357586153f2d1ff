"""The two routes of viscous stages (patch kernels; flux, viscous and gather kernels) agree bit for bit: triangles,
quadrilaterals, six-faced cells (no patch tables), tetrahedra, periodic faces, a boundary of unknown type, both
orders and precisions."""
import numpy as np
import pytest

import mstcfd as M
from helpers import brick_grid, cons, quad_grid

pytestmark = pytest.mark.gpu


def unknown_side():
    raw = M.Mesh.gen_tri(30, 20, 0, 3, 0, 2, 0.15, 7, (M.BC_INLET, M.BC_OUTLET, M.BC_WALL, M.BC_SYMMETRY)).raw()
    raw["ftype"][raw["ftype"] == M.BC_SYMMETRY] = 36  # no Fluent type the solver knows: no convective flux
    return M.Mesh.from_raw(raw)


MESHES = {
    "tri": lambda: M.Mesh.gen_tri(61, 40, 0, 3, 0, 2, 0.15, 7, (M.BC_INLET, M.BC_OUTLET, M.BC_WALL, M.BC_SYMMETRY)),
    "periodic": lambda: M.Mesh.gen_tri(24, 24, -1, 1, -1, 1, 0.15, 3, (M.BC_PERIODIC,) * 4),
    "quad": lambda: M.Mesh.from_raw(quad_grid(20, bc=M.BC_WALL, h=0.05, jitter=0.2, seed=4)),
    "brick": lambda: M.Mesh.from_raw(brick_grid(24, 20, h=0.05, jitter=0.1, seed=5, bc=M.BC_WALL)),
    "tet": lambda: M.Mesh.gen_tet(9, 8, 7, (0, 0, 0), (1, 0.8, 0.7), 0.15, 11,
                                  (M.BC_INLET, M.BC_OUTLET, M.BC_SYMMETRY, M.BC_WALL, M.BC_SYMMETRY, M.BC_WALL)),
    "unknown": unknown_side,
}


@pytest.mark.parametrize("order,prec", [(1, M.PREC_FP64), (2, M.PREC_FP64), (1, M.PREC_MIXED), (2, M.PREC_MIXED)])
@pytest.mark.parametrize("name", sorted(MESHES))
def test_routes_agree(name, order, prec):
    m = MESHES[name]()
    print(f"viscous routes {name}: {m.n_cells} cells, order {order}, precision {prec}", flush=True)
    rng = np.random.default_rng(3)
    n = m.n_cells
    Q = cons(rng.uniform(0.95, 1.05, n), rng.uniform(-0.1, 0.1, (n, m.dim)), rng.uniform(0.95, 1.05, n))
    out = []
    for st in (M.STRATEGY_FACE, M.STRATEGY_CELL, M.STRATEGY_AUTO):
        for scheme, lim in ((M.ROE, M.LIM_VANLEER), (M.AUSM, M.LIM_NONE)):
            s = M.Solver(m, M.make_config(dim=m.dim, scheme=scheme, order=order, limiter=lim, rk=3, precision=prec, mu=0.03,
                                          kappa=0.05, cv=2.5, q_inlet=list(Q[0])))
            s.strategy = st
            s.set_state(Q)
            s.set_dt(1e-4)
            s.step(2)
            out.append((s.get_state(), s.residual_norms()))
            s.close()
    for k, (q, r) in enumerate(out):
        assert np.all(np.isfinite(q))
        assert np.array_equal(q, out[k % 2][0]) and np.array_equal(r, out[k % 2][1])
